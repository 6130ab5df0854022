"""Gradients of gradients, with tensor operations on the CPU standing in for the kernels: what the formulas give must be what
differentiating the plain computation twice gives, and what they do not cover must be an error rather than zero."""

import pytest
import torch

import torch_ggml_ops as tgo
from torch_ggml_ops import _validate


def plain_combine(rows, slot_rows, slot_weights):
    present = (slot_rows >= 0) & (slot_rows < rows.shape[0])
    picked = rows[slot_rows.clamp(0, rows.shape[0] - 1)]
    return (picked * (slot_weights * present).unsqueeze(-1)).sum(1)


def plain_weight_grad(rows, grad_tokens, slot_rows):
    present = (slot_rows >= 0) & (slot_rows < rows.shape[0])
    return (rows[slot_rows.clamp(0, rows.shape[0] - 1)] * grad_tokens.unsqueeze(1)).sum(-1) * present


@pytest.fixture
def stand_ins():
    """Registers CPU implementations of the named operators for the time of a test."""
    library = torch.library.Library("torch_ggml_ops", "IMPL")

    def register(**implementations):
        for name, implementation in implementations.items():
            library.impl(name, torch.no_grad()(implementation), "CPU")   # (like a kernel: autograd sees nothing of it)

    yield register
    library._destroy()


@pytest.fixture
def combine_on_cpu(stand_ins):
    stand_ins(moe_combine=plain_combine, moe_combine_weight_grad=plain_weight_grad)


# (one slot past the rows, one before them, a row that no slot names)
SLOT_ROWS = torch.tensor([[0, 4], [7, 2], [3, -1]])


def combine_inputs():
    generator = torch.Generator().manual_seed(1)
    rows = torch.randn(6, 8, generator=generator).requires_grad_()
    weights = torch.rand(3, 2, generator=generator).requires_grad_()
    return rows, weights, torch.randn(3, 8, generator=generator).requires_grad_(), torch.randn(3, 2, generator=generator)


def test_gradients_of_the_routing_weights_gradient(combine_on_cpu):
    results = []
    for combine in (tgo.moe_combine, plain_combine):
        rows, weights, cotangent, direction = combine_inputs()
        (grad_weights,) = torch.autograd.grad(combine(rows, SLOT_ROWS, weights), weights, cotangent, create_graph=True)
        penalty = (grad_weights.square() * direction).sum()
        grad_rows, grad_cotangent = torch.autograd.grad(penalty, (rows, cotangent), create_graph=True)
        third = torch.autograd.grad(grad_rows.square().sum() + grad_cotangent.square().sum(), (rows, cotangent))
        results.append((grad_weights, grad_rows, grad_cotangent, *third))
    for actual, expected in zip(*results):
        assert expected.norm() > 0
        torch.testing.assert_close(actual, expected)   # (fp32 on both sides)


def test_gradient_through_the_expert_sorted_rows_is_refused(stand_ins, combine_on_cpu):
    """``grouped_mmq_combine`` has no gradient for what flows back through the sorted rows that its weights' gradient is
    made of: an error, not a part that is missing."""

    def product(input, packed, indices, offsets, slot_rows, slot_weights, quant_type, out_features):
        rows = input @ packed.float()
        return plain_combine(rows, slot_rows, slot_weights), rows

    stand_ins(grouped_mmq_combine=product)
    rows, weights, cotangent, _ = combine_inputs()
    packed = torch.randint(0, 3, (8, 8), generator=torch.Generator().manual_seed(2), dtype=torch.uint8)
    none = torch.zeros(1, dtype=torch.int64)
    out = tgo.grouped_mmq_combine(rows.detach(), packed, none, none, SLOT_ROWS, weights, 12, 8)
    (grad_weights,) = torch.autograd.grad(out, weights, cotangent, create_graph=True)
    with pytest.raises(RuntimeError, match="auxiliary output without a gradient"):
        grad_weights.sum().backward()


@pytest.mark.parametrize("widths", ((3, 5), (3, 3), (5, 3, 3)))
def test_projections_of_one_input_refuse_a_second_gradient(stand_ins, monkeypatch, widths):
    """Two neighbours of one shape and format share a grad-input kernel, the others have one each: both refuse alike."""
    monkeypatch.setattr(_validate, "REQUIRE_DEVICE", False)

    def product(grad, packed, quant_type, in_features):
        return (grad.float() @ packed.float()).to(grad.dtype)

    stand_ins(
        mmq_multi_forward=lambda input, weights, *rest: [(input.float() @ w.float().t()).to(input.dtype) for w in weights],
        mmq_grad_input=product,
        mmq_pair_grad_input=lambda g1, g2, w1, w2, *rest: product(g1, w1, *rest) + product(g2, w2, *rest),
    )
    generator = torch.Generator().manual_seed(3)
    x = torch.randn(4, 256, generator=generator).bfloat16().requires_grad_()
    weights = [torch.randint(0, 3, (n, 256), generator=generator, dtype=torch.uint8) for n in widths]
    outputs = tgo.mmq_multi(x, weights, [12] * len(widths), widths)
    cotangents = [torch.randn(o.shape, generator=generator).bfloat16().requires_grad_() for o in outputs]
    (grad,) = torch.autograd.grad(outputs, x, cotangents, create_graph=True)
    expected = sum(c.double() @ w.double() for c, w in zip(cotangents, weights))
    torch.testing.assert_close(grad.double(), expected, rtol=2**-6, atol=2**-6 * expected.abs().max().item())
    with pytest.raises(RuntimeError, match="does not support higher-order gradients"):
        torch.autograd.grad(grad.float().sum(), cotangents)


def _opaque(shape):
    return lambda *args, **kwargs: torch.ones(shape, dtype=torch.bfloat16)


@pytest.mark.parametrize("which", ("gathered", "pair_gathered", "swiglu", "swiglu_slots", "combine"))
def test_backward_made_of_kernels_refuses_a_second_gradient(stand_ins, combine_on_cpu, monkeypatch, which):
    """Backward formulas that call kernels directly: autograd sees a constant there, so what flows through it has to raise."""
    from torch_ggml_ops import gathered, swiglu

    rows, tokens, k, n = 6, 3, 256, 8
    generator = torch.Generator().manual_seed(4)
    hidden = torch.randn(tokens, k, generator=generator).bfloat16().requires_grad_()
    slot_weights = torch.rand(tokens, 2, generator=generator).requires_grad_()
    slot_rows = torch.arange(rows).reshape(tokens, 2)
    row_index = torch.arange(rows) // 2
    packed, ids = torch.zeros(1, n, 144, dtype=torch.uint8), torch.zeros(1, dtype=torch.int64)
    for module in (gathered, swiglu):
        monkeypatch.setattr(module, "_rows_grad_input", _opaque((rows, k)))
        monkeypatch.setattr(module, "_scatter_to_tokens", _opaque((tokens, k)))
    monkeypatch.setattr(swiglu, "_sum_slots", _opaque((tokens, k)))
    monkeypatch.setattr(swiglu, "_activation_backward", lambda *args: (torch.ones(rows, n, dtype=torch.bfloat16),) * 2)
    one = _opaque((rows, n))
    stand_ins(
        grouped_mmq_gathered=one,
        grouped_mmq_pair_gathered=lambda *args: (one(), one()),
        grouped_mmq_swiglu=lambda *args: (one(), one(), one()),
        grouped_mmq_combine=lambda *args: (torch.ones(tokens, n, dtype=torch.bfloat16), one()),
        invert_slots=lambda slot_rows, slot_weights, num_rows: (row_index.clone(), slot_weights.reshape(-1).clone()),
        grouped_mmq_grad_input_weighted=_opaque((tokens, k)),
    )
    if which == "gathered":
        outputs = (tgo.grouped_mmq_gathered(hidden, row_index, packed, ids, ids, 12, n),)
    elif which == "pair_gathered":
        outputs = tgo.grouped_mmq_pair_gathered(hidden, row_index, packed, packed, ids, ids, 12, n)
    elif which == "combine":
        outputs = (tgo.grouped_mmq_combine(hidden, packed, ids, ids, slot_rows, slot_weights, 12, n),)
    else:
        listed = slot_rows if which == "swiglu_slots" else None
        outputs = (tgo.grouped_mmq_swiglu(hidden, packed, packed, ids, ids, 12, n, row_index, listed),)
    cotangents = [torch.ones_like(o) for o in outputs]
    assert not torch.autograd.grad(outputs, hidden, cotangents, retain_graph=True)[0].requires_grad
    cotangents = [c.requires_grad_() for c in cotangents]
    (grad,) = torch.autograd.grad(outputs, hidden, cotangents, create_graph=True)
    penalty = grad.float().square().sum() + sum(c.float().sum() for c in cotangents)
    with pytest.raises(RuntimeError, match="does not support higher-order gradients"):
        torch.autograd.grad(penalty, cotangents)
