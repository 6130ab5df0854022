"""The steps of a mixture-of-experts layer on either side of the grouped operators.

The reference's grouped operators start and end at expert-sorted rows and leave routing to the
caller (torch_ggml_ops/grouped_mmq.py:216).  This module holds the caller's side for this library:

* ``route``        sorts the (token, choice) slots by expert without a host synchronisation,
* ``moe_combine``  returns sorted rows to tokens, ``out[t] = sum_j w[t, j] * rows[slot_rows[t, j]]``,
                   in one deterministic pass (fp32 accumulation in choice order, one rounding),
* ``grouped_mmq_combine``  is the down projection followed by ``moe_combine`` as one differentiable step: its
                   backward folds the gather and the routing-weight scaling of the combine's gradient into the
                   packing of the down projection's cotangent, so the expert-sorted cotangent is never built,
* ``moe_layer``    chains gathered gate/up pair with fused SwiGLU -> down + combine.
"""

from __future__ import annotations

import torch

from . import _native, _validate
from ._native import direct as _direct
from .grouped_mmq import _forward as _grouped_forward
from .grouped_mmq import _no_double_backward
from .swiglu import grouped_mmq_swiglu

torch.library.define(
    "torch_ggml_ops::moe_combine", "(Tensor rows, Tensor slot_rows, Tensor slot_weights) -> Tensor"
)


def _fail(message: str) -> None:
    raise RuntimeError(message)


def _check_combine(rows: torch.Tensor, slot_rows: torch.Tensor, slot_weights: torch.Tensor) -> None:
    for tensor, name in ((rows, "rows"), (slot_rows, "slot_rows"), (slot_weights, "slot_weights")):
        if not tensor.is_cuda:
            _fail(f"{name} must be a CUDA/HIP tensor")
        if tensor.device != rows.device:
            _fail("all moe_combine tensors must be on the same device")
        if not tensor.is_contiguous():
            _fail(f"{name} must be contiguous; torch_ggml_ops will not insert a hidden copy")
    if rows.dtype != torch.bfloat16:
        _fail("rows must have dtype torch.bfloat16")
    if slot_rows.dtype != torch.int64:
        _fail("slot_rows must have dtype torch.int64")
    if slot_weights.dtype != torch.float32:
        _fail("slot_weights must have dtype torch.float32")
    if rows.dim() != 2 or rows.shape[0] <= 0:
        _fail("rows must have shape [rows, features] with at least one row")
    if slot_rows.dim() != 2 or slot_rows.shape != slot_weights.shape or slot_rows.numel() <= 0:
        _fail("slot_rows and slot_weights must both have shape [tokens, top_k]")
    if rows.shape[1] <= 0 or rows.shape[1] % 8 != 0:
        _fail(f"features must be a positive multiple of 8; got {rows.shape[1]}")
    if rows.data_ptr() % 16 != 0:
        _fail("rows data pointer must be 16-byte aligned")


def _combine_device(rows, slot_rows, slot_weights):
    _check_combine(rows, slot_rows, slot_weights)
    tokens, top_k = slot_rows.shape
    with _native.on_device(rows.device):
        output = rows.new_empty((tokens, rows.shape[1]))
        _native.check(
            _native.lib.tgo_moe_combine(
                rows.data_ptr(), slot_rows.data_ptr(), slot_weights.data_ptr(), output.data_ptr(),
                tokens, top_k, rows.shape[0], rows.shape[1], _native.stream_of(rows.device),
            )
        )
    return output


torch.library.impl("torch_ggml_ops::moe_combine", "CUDA")(_combine_device)


@torch.library.register_fake("torch_ggml_ops::moe_combine")
def _combine_fake(rows, slot_rows, slot_weights):
    return rows.new_empty((slot_rows.shape[0], rows.shape[1]))


torch.library.define(
    "torch_ggml_ops::moe_combine_weight_grad", "(Tensor rows, Tensor grad_tokens, Tensor slot_rows) -> Tensor"
)
torch.library.define(
    "torch_ggml_ops::invert_slots", "(Tensor slot_rows, Tensor slot_weights, int num_rows) -> (Tensor, Tensor)"
)


def _check_weight_grad(rows, grad_tokens, slot_rows) -> None:
    _validate.operand(rows, "rows", torch.bfloat16, rows.device)
    _validate.operand(grad_tokens, "grad_tokens", torch.bfloat16, rows.device)
    _validate.operand(slot_rows, "slot_rows", torch.int64, rows.device)
    if rows.dim() != 2 or rows.shape[0] <= 0:
        _fail("rows must have shape [rows, features] with at least one row")
    if slot_rows.dim() != 2 or slot_rows.numel() <= 0:
        _fail("slot_rows must have shape [tokens, top_k]")
    if grad_tokens.shape != (slot_rows.shape[0], rows.shape[1]):
        _fail("grad_tokens must have shape [tokens, features]")
    if rows.shape[1] <= 0 or rows.shape[1] % 8 != 0:
        _fail(f"features must be a positive multiple of 8; got {rows.shape[1]}")


@torch.library.impl("torch_ggml_ops::moe_combine_weight_grad", "CUDA")
def _weight_grad_device(rows, grad_tokens, slot_rows):
    """Gradient of the routing weights of ``moe_combine``: the dot product of each slot's row with its token's gradient."""
    _check_weight_grad(rows, grad_tokens, slot_rows)
    if grad_tokens.data_ptr() % 16 != 0:   # (a view into a larger gradient: autograd hands over whatever address that has)
        grad_tokens = grad_tokens.clone()
    tokens, top_k = slot_rows.shape
    grad_weights = torch.empty((tokens, top_k), dtype=torch.float32, device=rows.device)
    with _native.on_device(rows.device):
        _native.check(
            _native.lib.tgo_slot_weight_grad(
                rows.data_ptr(), grad_tokens.data_ptr(), slot_rows.data_ptr(), grad_weights.data_ptr(), tokens, top_k,
                rows.shape[0], rows.shape[1], _native.stream_of(rows.device),
            )
        )
    return grad_weights


@torch.library.register_fake("torch_ggml_ops::moe_combine_weight_grad")
def _weight_grad_fake(rows, grad_tokens, slot_rows):
    return slot_rows.new_empty(slot_rows.shape, dtype=torch.float32)


def _check_inverse(slot_rows, slot_weights, num_rows) -> None:
    _validate.operand(slot_rows, "slot_rows", torch.int64, slot_weights.device)
    _validate.operand(slot_weights, "slot_weights", torch.float32, slot_weights.device)
    if slot_rows.dim() != 2 or slot_rows.shape != slot_weights.shape or slot_rows.numel() <= 0:
        _fail("slot_rows and slot_weights must both have shape [tokens, top_k]")
    if num_rows <= 0:
        _fail(f"num_rows must be positive; got {num_rows}")


@torch.library.impl("torch_ggml_ops::invert_slots", "CUDA")
def _invert_slots_device(slot_rows, slot_weights, num_rows):
    """Token and routing weight of every expert-sorted row; -1 and 0 for a row that no slot names."""
    _check_inverse(slot_rows, slot_weights, num_rows)
    tokens, top_k = slot_rows.shape
    row_token = torch.empty(num_rows, dtype=torch.int64, device=slot_rows.device)
    row_weight = torch.empty(num_rows, dtype=torch.float32, device=slot_rows.device)
    with _native.on_device(slot_rows.device):
        _native.check(
            _native.lib.tgo_invert_slots(
                slot_rows.data_ptr(), slot_weights.data_ptr(), tokens, top_k, num_rows, row_token.data_ptr(),
                row_weight.data_ptr(), _native.stream_of(slot_rows.device),
            )
        )
    return row_token, row_weight


@torch.library.register_fake("torch_ggml_ops::invert_slots")
def _invert_slots_fake(slot_rows, slot_weights, num_rows):
    return slot_rows.new_empty((num_rows,)), slot_rows.new_empty((num_rows,), dtype=torch.float32)


def _slots_to_rows(grad_tokens, slot_rows, slot_weights, num_rows):
    """``out[slot_rows[t, j]] = slot_weights[t, j] * grad_tokens[t]``, zeros in the rows that no slot names."""
    flat = slot_rows.reshape(-1)
    present = (flat >= 0) & (flat < num_rows)
    per_slot = grad_tokens.repeat_interleave(slot_rows.shape[1], dim=0)
    scaled = (per_slot.float() * (slot_weights.reshape(-1, 1) * present.unsqueeze(1))).to(grad_tokens.dtype)
    out = grad_tokens.new_zeros((num_rows, grad_tokens.shape[1]))
    # every row belongs to at most one slot, so this is a plain scatter, not a reduction
    out.index_add_(0, flat.clamp(0, num_rows - 1), scaled)
    return out


def _setup_weight_grad_context(ctx, inputs, output) -> None:
    rows, grad_tokens, slot_rows = inputs
    ctx.num_rows = rows.shape[0]
    ctx.save_for_backward(
        rows if ctx.needs_input_grad[1] else None, grad_tokens if ctx.needs_input_grad[0] else None, slot_rows
    )


def _weight_grad_backward(ctx, grad):
    """The product is bilinear: the one factor's gradient is the combine with ``grad`` as its weights, the other's the
    combine's own backward."""
    rows, grad_tokens, slot_rows = ctx.saved_tensors
    grad_rows = grad_grad_tokens = None
    if ctx.needs_input_grad[0]:
        grad_rows = _slots_to_rows(grad_tokens, slot_rows, grad, ctx.num_rows)
    if ctx.needs_input_grad[1]:
        grad_grad_tokens = torch.ops.torch_ggml_ops.moe_combine.default(rows, slot_rows, grad.contiguous())
    return grad_rows, grad_grad_tokens, None


torch.library.register_autograd(
    "torch_ggml_ops::moe_combine_weight_grad", _weight_grad_backward, setup_context=_setup_weight_grad_context
)


def _setup_combine_context(ctx, inputs, output) -> None:
    rows, slot_rows, slot_weights = inputs
    ctx.num_rows = rows.shape[0]
    ctx.save_for_backward(rows if ctx.needs_input_grad[2] else None, slot_rows, slot_weights)


def _combine_backward(ctx, grad_output):
    rows, slot_rows, slot_weights = ctx.saved_tensors
    grad_rows = grad_weights = None
    if ctx.needs_input_grad[0]:
        grad_rows = _slots_to_rows(grad_output, slot_rows, slot_weights, ctx.num_rows)
    if ctx.needs_input_grad[2]:
        grad_weights = torch.ops.torch_ggml_ops.moe_combine_weight_grad.default(rows, grad_output.contiguous(), slot_rows)
    return grad_rows, None, grad_weights


torch.library.register_autograd("torch_ggml_ops::moe_combine", _combine_backward, setup_context=_setup_combine_context)


def moe_combine(rows: torch.Tensor, slot_rows: torch.Tensor, slot_weights: torch.Tensor) -> torch.Tensor:
    """``out[t] = sum_j slot_weights[t, j] * rows[slot_rows[t, j]]``: bf16 rows, fp32 weights, bf16 result."""
    return torch.ops.torch_ggml_ops.moe_combine.default(rows, slot_rows, slot_weights)


torch.library.define(
    "torch_ggml_ops::grouped_mmq_grad_input_weighted",
    "(Tensor grad_tokens, Tensor row_token, Tensor row_weight, Tensor packed_weight, Tensor expert_indices, "
    "Tensor expert_offsets, int quant_type, int in_features) -> Tensor",
)
torch.library.define(
    "torch_ggml_ops::grouped_mmq_combine",
    "(Tensor input, Tensor packed_weight, Tensor expert_indices, Tensor expert_offsets, Tensor slot_rows, "
    "Tensor slot_weights, int quant_type, int out_features) -> (Tensor, Tensor)",
)


@torch.library.impl("torch_ggml_ops::grouped_mmq_grad_input_weighted", "CUDA")
def _grad_input_weighted_device(
    grad_tokens, row_token, row_weight, packed_weight, expert_indices, expert_offsets, quant_type, in_features
):
    shape = _validate.grouped(
        grad_tokens, packed_weight, expert_indices, expert_offsets, quant_type, in_features, backward=True
    )
    tokens, in_features, out_features, experts, groups, _bytes_per_expert = shape
    rows = _validate.row_index(row_token, grad_tokens)
    if row_weight.dtype != torch.float32 or row_weight.shape != row_token.shape or not row_weight.is_contiguous():
        _fail("row_weight must be a contiguous torch.float32 tensor with one entry per row")
    if row_weight.device != grad_tokens.device:
        _fail("all grouped MMQ backward tensors must be on the same device")
    with _native.on_device(grad_tokens.device):
        # (rows that no valid group covers stay unwritten, as for grouped_mmq_grad_input)
        grad_input = grad_tokens.new_empty((rows, in_features))
        workspace = grad_tokens.new_empty(
            (_native.lib.tgo_grad_workspace_bytes(rows, out_features, groups, 1),), dtype=torch.uint8
        )
        _native.check(
            _native.lib.tgo_grouped_mmq_grad_input_weighted(
                grad_tokens.data_ptr(), row_token.data_ptr(), row_weight.data_ptr(), tokens,
                packed_weight.data_ptr(), grad_input.data_ptr(), expert_indices.data_ptr(), expert_offsets.data_ptr(),
                workspace.data_ptr(), rows, out_features, in_features, experts, groups, int(quant_type),
                _native.stream_of(grad_tokens.device),
            )
        )
    return grad_input


@torch.library.register_fake("torch_ggml_ops::grouped_mmq_grad_input_weighted")
def _grad_input_weighted_fake(
    grad_tokens, row_token, row_weight, packed_weight, expert_indices, expert_offsets, quant_type, in_features
):
    return grad_tokens.new_empty((row_token.shape[0], in_features))


torch.library.register_autograd(
    "torch_ggml_ops::grouped_mmq_grad_input_weighted", _no_double_backward("grouped_mmq_grad_input_weighted")
)


@torch.library.impl("torch_ggml_ops::grouped_mmq_combine", "CUDA")
def _grouped_combine_device(
    input, packed_weight, expert_indices, expert_offsets, slot_rows, slot_weights, quant_type, out_features
):
    rows = _grouped_forward(input, packed_weight, None, expert_indices, expert_offsets, quant_type, out_features)[0]
    return _combine_device(rows, slot_rows, slot_weights), rows


@torch.library.register_fake("torch_ggml_ops::grouped_mmq_combine")
def _grouped_combine_fake(
    input, packed_weight, expert_indices, expert_offsets, slot_rows, slot_weights, quant_type, out_features
):
    return input.new_empty((slot_rows.shape[0], out_features)), input.new_empty((input.shape[0], out_features))


def _setup_grouped_combine_context(ctx, inputs, output) -> None:
    input, packed_weight, expert_indices, expert_offsets, slot_rows, slot_weights, quant_type, _out_features = inputs
    ctx.quant_type = quant_type
    ctx.num_rows, ctx.in_features = input.shape
    # (the second output, the expert-sorted rows, only serves the gradient of the routing weights: without this the
    # engine would hand the backward a zero tensor of its size)
    ctx.set_materialize_grads(False)
    ctx.save_for_backward(
        packed_weight, expert_indices, expert_offsets, slot_rows, slot_weights,
        output[1] if ctx.needs_input_grad[5] else None,
    )


def _grouped_combine_backward(ctx, grad_output, grad_rows):
    if grad_rows is not None:
        raise RuntimeError("grouped_mmq_combine: the expert-sorted rows are an auxiliary output without a gradient")
    packed_weight, expert_indices, expert_offsets, slot_rows, slot_weights, rows = ctx.saved_tensors
    if grad_output is None:
        return None, None, None, None, None, None, None, None
    grad_output = grad_output.contiguous()
    grad_input = grad_weights = None
    if ctx.needs_input_grad[0]:
        # the inverse of slot_rows: token and routing weight of every expert-sorted row (rows that no slot names
        # have token -1, i.e. a zero cotangent)
        row_token, row_weight = torch.ops.torch_ggml_ops.invert_slots.default(slot_rows, slot_weights, ctx.num_rows)
        grad_input = torch.ops.torch_ggml_ops.grouped_mmq_grad_input_weighted.default(
            grad_output, row_token, row_weight, packed_weight, expert_indices, expert_offsets, ctx.quant_type, ctx.in_features
        )
    if ctx.needs_input_grad[5]:
        grad_weights = torch.ops.torch_ggml_ops.moe_combine_weight_grad.default(rows, grad_output, slot_rows)
    return grad_input, None, None, None, None, grad_weights, None, None


torch.library.register_autograd(
    "torch_ggml_ops::grouped_mmq_combine", _grouped_combine_backward, setup_context=_setup_grouped_combine_context
)


def grouped_mmq_combine(
    input: torch.Tensor,
    packed_weight: torch.Tensor,
    expert_indices: torch.Tensor,
    expert_offsets: torch.Tensor,
    slot_rows: torch.Tensor,
    slot_weights: torch.Tensor,
    quant_type: int,
    out_features: int,
) -> torch.Tensor:
    """``moe_combine(grouped_mmq(input, packed_weight, ...), slot_rows, slot_weights)`` as one differentiable step.

    Forward: the grouped projection of the expert-sorted ``input`` rows, then the routing-weighted return to
    tokens (bit-identical to the two separate calls).  Backward with respect to ``input``: the per-token gradient
    is gathered and scaled by the routing weight while the projection's cotangent is packed, so the
    expert-sorted gradient of the separate calls (``rows x out_features`` bf16 written, then read) never exists;
    the result equals theirs bit for bit.  Also differentiable with respect to ``slot_weights``.

    Every expert-sorted row may be named by at most one (token, choice) slot of ``slot_rows``, as ``route``
    guarantees: the backward inverts ``slot_rows`` into one (token, weight) per row, so a row named twice would keep
    one of its slots only, whereas the forward (and the separate ``moe_combine``) adds both.
    """
    output, _rows = torch.ops.torch_ggml_ops.grouped_mmq_combine.default(
        input, packed_weight, expert_indices, expert_offsets, slot_rows, slot_weights, int(quant_type), int(out_features)
    )
    return output


ROUTE_SLOT_LIMIT = 4194304   # TGO_ROUTE_SLOT_LIMIT
ROUTE_EXPERT_LIMIT = 4096    # TGO_ROUTE_EXPERT_LIMIT


for _name in ("route", "route_small"):
    torch.library.define(
        f"torch_ggml_ops::{_name}", "(Tensor slot_experts, int num_experts) -> (Tensor, Tensor, Tensor, Tensor)"
    )


def _route_outputs(slot_experts, num_experts):
    tokens, top_k = slot_experts.shape
    return (
        slot_experts.new_empty((tokens * top_k,), dtype=torch.int64),
        slot_experts.new_empty((tokens, top_k), dtype=torch.int64),
        slot_experts.new_empty((num_experts,), dtype=torch.int64),
        slot_experts.new_empty((num_experts,), dtype=torch.int32),
    )


@torch.library.impl("torch_ggml_ops::route", "CUDA")
def _route_device(slot_experts, num_experts):
    """``route`` as one or two kernels (``tgo_route``) instead of a sort and a dozen tensor operations, which cost more
    than a layer's own launches at decode sizes and a third of its time in a prefill.  Same results."""
    slot_experts = slot_experts.to(torch.int64).contiguous()
    tokens, top_k = slot_experts.shape
    device = slot_experts.device
    outputs = _route_outputs(slot_experts, num_experts)
    workspace_bytes = _native.lib.tgo_route_workspace_bytes(tokens * top_k, num_experts)
    workspace = torch.empty(workspace_bytes, dtype=torch.uint8, device=device) if workspace_bytes > 0 else None
    with _native.on_device(device):
        _native.check(
            _native.lib.tgo_route(
                slot_experts.data_ptr(), tokens, top_k, num_experts, *(output.data_ptr() for output in outputs),
                None if workspace is None else workspace.data_ptr(), _native.stream_of(device),
            )
        )
    return outputs


@torch.library.impl("torch_ggml_ops::route_small", "CUDA")
def _route_small_device(slot_experts, num_experts):
    """``route`` for a batch of one launch, which needs no workspace (at most 4096 slots and experts)."""
    slot_experts = slot_experts.to(torch.int64).contiguous()
    tokens, top_k = slot_experts.shape
    outputs = _route_outputs(slot_experts, num_experts)
    with _native.on_device(slot_experts.device):
        _native.check(
            _native.lib.tgo_route_small(
                slot_experts.data_ptr(), tokens, top_k, num_experts, *(output.data_ptr() for output in outputs),
                _native.stream_of(slot_experts.device),
            )
        )
    return outputs


for _name in ("route", "route_small"):
    torch.library.register_fake(f"torch_ggml_ops::{_name}")(_route_outputs)


def route(slot_experts: torch.Tensor, num_experts: int):
    """Sorts the ``[tokens, top_k]`` expert choices by expert (stable, no host synchronisation).

    Returns ``(row_index, slot_rows, expert_indices, expert_offsets)``: the token of each sorted row, the
    sorted row of each (token, choice) slot, and the group metadata of the grouped operators with one
    group per expert (experts without rows are empty groups, which the operators skip).
    """
    tokens, top_k = slot_experts.shape
    if slot_experts.is_cuda and 0 < tokens * top_k <= ROUTE_SLOT_LIMIT and 0 < num_experts <= ROUTE_EXPERT_LIMIT:
        return torch.ops.torch_ggml_ops.route.default(slot_experts, int(num_experts))
    flat = slot_experts.reshape(-1)
    order = torch.argsort(flat, stable=True)
    row_index = torch.div(order, top_k, rounding_mode="floor")
    slot_rows = torch.empty_like(order)
    slot_rows[order] = torch.arange(order.numel(), device=order.device)
    counts = torch.zeros(num_experts, dtype=torch.int64, device=flat.device)
    counts.scatter_add_(0, flat, torch.ones_like(flat))
    expert_offsets = counts.cumsum(0).to(torch.int32)
    expert_indices = torch.arange(num_experts, dtype=torch.int64, device=flat.device)
    return row_index, slot_rows.reshape(tokens, top_k), expert_indices, expert_offsets


def moe_layer(
    hidden: torch.Tensor,
    slot_experts: torch.Tensor,
    slot_weights: torch.Tensor,
    gate_weight: torch.Tensor,
    up_weight: torch.Tensor,
    down_weight: torch.Tensor,
    gate_up_type: int,
    down_type: int,
    intermediate_features: int,
) -> torch.Tensor:
    """SwiGLU mixture-of-experts layer over packed expert weights.

    ``hidden`` bf16 ``[tokens, features]``; ``slot_experts`` int64 and ``slot_weights`` fp32
    ``[tokens, top_k]``; ``gate_weight``/``up_weight`` packed ``[experts, intermediate, ...]`` and
    ``down_weight`` packed ``[experts, features, ...]``.  Differentiable with respect to ``hidden`` and
    ``slot_weights``.

    A plain call without a gradient for a few tokens (up to 64 choices of experts of a decode step's sizes) is two launches
    of their own and gives other bits than the same call with a gradient, or under a mode or a tracer: it rounds the sum over a token's
    experts once, where the operators round every expert's row first.
    """
    if _direct is not None and not torch.compiler.is_compiling():
        output = _direct.moe_layer(
            hidden, slot_experts, slot_weights, gate_weight, up_weight, down_weight, gate_up_type, down_type,
            intermediate_features,
        )   # (None: not a plain call)
        if output is not None:
            return output
    experts = gate_weight.shape[0]
    row_index, slot_rows, expert_indices, expert_offsets = route(slot_experts, experts)
    activated = grouped_mmq_swiglu(
        hidden, gate_weight, up_weight, expert_indices, expert_offsets, gate_up_type, intermediate_features, row_index,
        slot_rows,
    )
    return grouped_mmq_combine(
        activated, down_weight, expert_indices, expert_offsets, slot_rows, slot_weights, down_type, hidden.shape[1]
    )


__all__ = ["grouped_mmq_combine", "moe_combine", "moe_layer", "route"]
