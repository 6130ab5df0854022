"""Cross-entropy through a packed LM head, one chunk of rows at a time.

The logits of an LM head are ``rows x vocabulary`` (248 320 columns for the model family the
reference is tuned on); keeping them for the backward pass of the loss costs more memory than
the rest of the step.  The reference's production schedule therefore walks the rows in chunks of
256 (its measured best; 128 and 64 are its lower-memory fallbacks,
docs/mmq_fwd_optimization.md:293) and runs forward and backward of each chunk back to back:
the forward product for the chunk's logits, the loss and its gradient with respect to the logits, and
the grad-input product for the chunk's share of the hidden-state gradient.  Only one chunk of logits
exists at a time.  That loop lives in the reference's training code, not in its package; here it is one
call into the library, whose loss kernels write the logits' gradient as the operand the grad-input kernels
read.
"""

from __future__ import annotations

import torch

from . import _native, _validate

DEFAULT_CHUNK_ROWS = 256   # the reference's production chunk


torch.library.define(
    "torch_ggml_ops::lm_head_loss",
    "(Tensor hidden, Tensor packed_weight, Tensor targets, int quant_type, int out_features, int chunk_rows, "
    "int ignore_index, bool gradient) -> (Tensor, Tensor)",
)


def _check_loss(hidden, targets, chunk_rows) -> None:
    if hidden.dim() != 2:
        raise RuntimeError("hidden must have shape [rows, in_features]")
    if targets.dim() != 1 or targets.shape[0] != hidden.shape[0] or targets.dtype != torch.int64:
        raise RuntimeError("targets must be an int64 tensor with one entry per row of hidden")
    if chunk_rows <= 0:
        raise RuntimeError("chunk_rows must be positive")


@torch.library.impl("torch_ggml_ops::lm_head_loss", "CUDA")
def _lm_head_loss_device(hidden, packed_weight, targets, quant_type, out_features, chunk_rows, ignore_index, gradient):
    """(mean loss, its gradient with respect to ``hidden`` or an empty tensor): every launch of every chunk is issued by
    one call into the library (``tgo_lm_head_loss``)."""
    _check_loss(hidden, targets, chunk_rows)
    if hidden.shape[0] > chunk_rows and (not hidden.is_contiguous() or hidden.storage_offset() != 0):
        hidden = hidden.clone(memory_format=torch.contiguous_format)   # (such rows were always accepted chunk by chunk)
    rows, in_features, out_features = _validate.dense(hidden, packed_weight, quant_type, out_features, backward=False)
    targets = targets.contiguous()
    if targets.device != hidden.device:
        raise RuntimeError("hidden and targets must be on the same device")
    with _native.on_device(hidden.device):
        loss = torch.empty((), dtype=torch.float32, device=hidden.device)
        grad_hidden = torch.empty_like(hidden) if gradient else hidden.new_empty((0, in_features))
        workspace_bytes = _native.lib.tgo_lm_head_workspace_bytes(
            rows, in_features, out_features, chunk_rows, int(quant_type), int(gradient)
        )
        workspace = torch.empty(max(workspace_bytes, 0), dtype=torch.uint8, device=hidden.device)
        _native.check(
            _native.lib.tgo_lm_head_loss(
                hidden.data_ptr(), packed_weight.data_ptr(), targets.data_ptr(), loss.data_ptr(),
                grad_hidden.data_ptr() if gradient else None, workspace.data_ptr(), rows, in_features, out_features,
                chunk_rows, ignore_index, int(quant_type), _native.stream_of(hidden.device),
            )
        )
    return loss, grad_hidden


@torch.library.register_fake("torch_ggml_ops::lm_head_loss")
def _lm_head_loss_fake(hidden, packed_weight, targets, quant_type, out_features, chunk_rows, ignore_index, gradient):
    return (
        hidden.new_empty((), dtype=torch.float32), hidden.new_empty(hidden.shape if gradient else (0, hidden.shape[1]))
    )


torch.library.define("torch_ggml_ops::scale_bf16", "(Tensor input, Tensor factor) -> Tensor")


def _check_scale(input, factor) -> None:
    _validate.operand(input, "input", torch.bfloat16, input.device)
    _validate.operand(factor, "factor", torch.float32, input.device)
    if factor.numel() != 1:
        raise RuntimeError("factor must have one element")


@torch.library.impl("torch_ggml_ops::scale_bf16", "CUDA")
def _scale_device(input, factor):
    """``(input.float() * factor).to(bfloat16)`` for a contiguous bf16 tensor and an fp32 scalar on its device."""
    _check_scale(input, factor)
    out = torch.empty_like(input)
    with _native.on_device(input.device):
        _native.check(
            _native.lib.tgo_scale_bf16(
                input.data_ptr(), factor.data_ptr(), out.data_ptr(), input.numel(), _native.stream_of(input.device)
            )
        )
    return out


@torch.library.register_fake("torch_ggml_ops::scale_bf16")
def _scale_fake(input, factor):
    return input.new_empty(input.shape)


class _ChunkedLoss(torch.autograd.Function):
    @staticmethod
    def forward(ctx, hidden, packed_weight, targets, quant_type, out_features, chunk_rows, ignore_index):
        if hidden.shape[0] == 0:   # (no chunk, no launch: the loss of a batch without any counted row)
            if ctx.needs_input_grad[0]:
                ctx.save_for_backward(torch.empty_like(hidden))
            return torch.zeros((), dtype=torch.float32, device=hidden.device)
        loss, grad_hidden = torch.ops.torch_ggml_ops.lm_head_loss.default(
            hidden, packed_weight, targets, quant_type, out_features, chunk_rows, ignore_index, ctx.needs_input_grad[0]
        )
        if ctx.needs_input_grad[0]:
            ctx.save_for_backward(grad_hidden)
        return loss

    @staticmethod
    def backward(ctx, grad_loss):
        grad_hidden = None
        if ctx.needs_input_grad[0]:
            (saved,) = ctx.saved_tensors
            # (a gradient of the gradient: tensor operations, which autograd can follow; no rows: nothing to launch)
            if grad_loss.requires_grad or saved.shape[0] == 0:
                grad_hidden = (saved.float() * grad_loss).to(saved.dtype)
            else:
                grad_hidden = torch.ops.torch_ggml_ops.scale_bf16.default(saved, grad_loss)
        return grad_hidden, None, None, None, None, None, None


def chunked_lm_head_loss(
    hidden: torch.Tensor,
    packed_weight: torch.Tensor,
    targets: torch.Tensor,
    quant_type: int,
    out_features: int,
    chunk_rows: int = DEFAULT_CHUNK_ROWS,
    ignore_index: int = -100,
) -> torch.Tensor:
    """Mean cross-entropy of ``mmq(hidden, packed_weight)`` against ``targets`` over the rows whose target is
    not ``ignore_index``, computed ``chunk_rows`` rows at a time.

    ``hidden`` bf16 ``[rows, in_features]`` (contiguous), ``targets`` int64 ``[rows]``.  Differentiable with
    respect to ``hidden``: the gradient is computed chunk by chunk during the forward pass (each chunk's logits
    are dropped as soon as its grad-input product has run) and scaled by the incoming gradient in backward.
    Equals ``cross_entropy(mmq(hidden, ...).float(), targets)`` up to the bf16 rounding of the logit gradients.
    """
    _check_loss(hidden, targets, chunk_rows)
    return _ChunkedLoss.apply(
        hidden, packed_weight, targets, int(quant_type), int(out_features), int(chunk_rows), int(ignore_index)
    )


__all__ = ["DEFAULT_CHUNK_ROWS", "chunked_lm_head_loss"]
