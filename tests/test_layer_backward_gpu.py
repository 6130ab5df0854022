"""Kernels around the matrix products of a layer and of the loss at the sizes where they can go wrong (-m gpu): the
routing sort in one and in several workgroups, the gradient of the routing weights, the clearing of uncovered rows, and
the loss of a chunk whose vocabulary is no multiple of a piece, a span or a tile."""

import numpy as np
import pytest
import torch

from helpers import QTYPES, f32, nrmse, random_bf16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import torch_ggml_ops
    import synth

    assert torch.cuda.is_available()
    return torch_ggml_ops, synth


@pytest.mark.parametrize("slots,experts", ((4096, 256), (4097, 257), (5000, 4096), (65 * 1024 + 3, 1025), (200_001, 255), (70_000, 1)))
def test_route_in_several_workgroups(ops, slots, experts):
    """Stable sort by expert with slots whose expert does not exist: those get row -1 and the rows behind the last are -1."""
    tgo, _ = ops
    flat = np.random.default_rng(slots).integers(-1, experts + 1, size=slots)
    row_index, slot_rows, indices, offsets = tgo.route(torch.from_numpy(flat.reshape(slots, 1)).cuda(), experts)
    valid = (flat >= 0) & (flat < experts)
    order = np.argsort(np.where(valid, flat, experts), kind="stable")[: valid.sum()]
    assert np.array_equal(row_index.cpu().numpy()[: order.size], order)
    assert (row_index[order.size :] == -1).all()
    expected = np.full(slots, -1)
    expected[order] = np.arange(order.size)
    assert np.array_equal(slot_rows.reshape(-1).cpu().numpy(), expected)
    assert np.array_equal(offsets.cpu().numpy(), np.cumsum(np.bincount(flat[valid], minlength=experts)))
    assert np.array_equal(indices.cpu().numpy(), np.arange(experts))


@pytest.mark.parametrize("tokens,top_k,experts", ((1, 8, 256), (512, 8, 4096)))
def test_route_of_one_launch(ops, tokens, top_k, experts):
    tgo, _ = ops
    chosen = torch.randint(-1, experts + 1, (tokens, top_k), generator=torch.Generator().manual_seed(tokens)).cuda()
    small = torch.ops.torch_ggml_ops.route_small.default(chosen, experts)
    for actual, expected in zip(small, tgo.route(chosen, experts), strict=True):
        assert actual.dtype == expected.dtype and torch.equal(actual, expected)
    with pytest.raises(RuntimeError, match="at most 4096 slots"):
        torch.ops.torch_ggml_ops.route_small.default(chosen.repeat(4097, 1), experts)


@pytest.mark.parametrize("tokens,top_k,features", ((1, 1, 8), (5, 3, 520), (33, 8, 2048)))
def test_routing_weight_gradient_and_inverse(ops, tokens, top_k, features):
    tgo, _ = ops
    num_rows = tokens * top_k
    generator = np.random.default_rng(features)
    slots = generator.permutation(num_rows + 2)[: tokens * top_k] - 1   # one slot may be -1 and one past the rows
    slot_rows = torch.from_numpy(slots.reshape(tokens, top_k)).cuda()
    rows, grad = random_bf16((num_rows, features), seed=1), random_bf16((tokens, features), seed=2)
    weights = torch.rand(tokens, top_k, device="cuda")
    actual = torch.ops.torch_ggml_ops.moe_combine_weight_grad.default(rows, grad, slot_rows)
    present = (slots >= 0) & (slots < num_rows)
    picked = rows.double()[torch.from_numpy(np.where(present, slots, 0)).cuda()].reshape(tokens, top_k, features)
    expected = (picked * grad.double().unsqueeze(1)).sum(-1) * torch.from_numpy(present.reshape(tokens, top_k)).cuda()
    torch.testing.assert_close(actual.double(), expected, rtol=1e-5, atol=1e-4)
    token, weight = torch.ops.torch_ggml_ops.invert_slots.default(slot_rows, weights, num_rows)
    expected_token, expected_weight = np.full(num_rows, -1), np.zeros(num_rows, dtype=np.float32)
    for i in np.flatnonzero(present):
        expected_token[slots[i]], expected_weight[slots[i]] = i // top_k, weights.cpu().numpy().reshape(-1)[i]
    assert np.array_equal(token.cpu().numpy(), expected_token) and np.array_equal(weight.cpu().numpy(), expected_weight)


@pytest.mark.parametrize("offset", (0, 1, 8))
def test_routing_weight_gradient_of_a_view_at_any_address(ops, offset):
    """The gradient of a part of a concatenation is a view into the whole, at whatever address that part has."""
    tgo, _ = ops
    tokens, top_k, features = 5, 2, 24
    rows = random_bf16((tokens * top_k, features), seed=1).requires_grad_()
    slot_rows = torch.arange(tokens * top_k, device="cuda").reshape(tokens, top_k)
    weights = torch.rand(tokens, top_k, device="cuda").requires_grad_()
    ahead = torch.zeros(offset, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    cotangent = random_bf16((offset + tokens * features,), seed=2)
    joined = torch.cat((ahead, tgo.moe_combine(rows, slot_rows, weights).flatten()))
    grad_rows, grad_weights = torch.autograd.grad(joined, (rows, weights), cotangent)
    mine = cotangent[offset:].reshape(tokens, 1, features).double()
    expected = (rows.detach().double().reshape(tokens, top_k, features) * mine).sum(-1)
    torch.testing.assert_close(grad_weights.double(), expected, rtol=1e-5, atol=1e-4)
    expected = (mine * weights.detach().double().unsqueeze(-1)).reshape(-1, features)
    torch.testing.assert_close(grad_rows.double(), expected, rtol=2**-8, atol=1e-6)


def test_gradients_of_the_routing_weight_gradient(ops):
    tgo, _ = ops
    tokens, top_k, features = 33, 4, 72
    slot_rows = torch.randperm(tokens * top_k, generator=torch.Generator().manual_seed(1)).reshape(tokens, top_k).cuda()
    slot_rows[0, 1], slot_rows[5, 0] = -1, tokens * top_k
    results = []
    for dtype in (torch.bfloat16, torch.float64):
        rows = random_bf16((tokens * top_k, features), seed=2).to(dtype).requires_grad_()
        cotangent = random_bf16((tokens, features), seed=3).to(dtype).requires_grad_()
        weights = torch.ones(tokens, top_k, device="cuda", requires_grad=True)
        if dtype == torch.bfloat16:
            out = tgo.moe_combine(rows, slot_rows, weights)
        else:
            present = (slot_rows >= 0) & (slot_rows < tokens * top_k)
            out = (rows[slot_rows.clamp(0, tokens * top_k - 1)] * (weights * present).unsqueeze(-1)).sum(1)
        (grad_weights,) = torch.autograd.grad(out, weights, cotangent, create_graph=True)
        results.append(torch.autograd.grad(grad_weights.square().sum(), (rows, cotangent)))
    for actual, expected in zip(*results):
        # (each result is rounded to bf16 once)
        torch.testing.assert_close(actual.double(), expected, rtol=2**-8, atol=1e-4 * expected.abs().max().item())


@pytest.mark.parametrize("rows,offsets,experts", ((700, (3, 3, 255, 256, 600), (0, 1, 7, 2, 3)), (5, (5,), (0,)), (300, (400, 10), (0, 1))))
def test_rows_outside_every_group_are_cleared(ops, rows, offsets, experts):
    """Empty groups, groups of an expert that does not exist and groups that end behind the rows cover nothing."""
    from torch_ggml_ops import _native

    x = torch.ones(rows, 24, dtype=torch.bfloat16, device="cuda")
    indices = torch.tensor(experts, dtype=torch.int64, device="cuda")
    ends = torch.tensor(offsets, dtype=torch.int32, device="cuda")
    _native.check(_native.lib.tgo_clear_uncovered_rows(
        x.data_ptr(), rows, 24, indices.data_ptr(), ends.data_ptr(), 5, len(offsets), torch.cuda.current_stream().cuda_stream))
    covered, begin = np.zeros(rows, dtype=bool), 0
    for end, expert in zip(offsets, experts):
        if begin < end <= rows and expert < 5:
            covered[begin:end] = True
        begin = end
    assert np.array_equal(x.float().cpu().numpy(), np.broadcast_to(covered[:, None], (rows, 24)).astype(np.float32))


def test_swiglu_with_slot_rows_equals_the_sorted_gradient(ops):
    tgo, synth = ops
    tokens, top_k, experts, k, n = 70, 3, 5, 512, 64
    gate, up = (synth.random_packed_weight(12, (experts, n), k, seed=s).cuda() for s in (1, 2))
    slot_experts = torch.from_numpy(np.random.default_rng(3).integers(0, experts, size=(tokens, top_k))).cuda()
    row_index, slot_rows, indices, offsets = tgo.route(slot_experts, experts)
    grads = []
    for listed in (None, slot_rows):
        hidden = random_bf16((tokens, k), seed=4).requires_grad_(True)
        out = tgo.grouped_mmq_swiglu(hidden, gate, up, indices, offsets, 12, n, row_index, listed)
        out.backward(random_bf16(out.shape, seed=5))
        grads.append(hidden.grad)
    assert nrmse(f32(grads[1]), f32(grads[0])) < 3e-3   # (the order of the fp32 sums of a token's rows)


@pytest.mark.parametrize("qname,rows,vocabulary,chunk", (("Q6_K", 70, 8195, 64), ("Q4_K", 33, 1001, 32), ("Q5_K", 3, 40, 256), ("Q6_K", 300, 33000, 256)))
def test_loss_of_ragged_vocabularies(ops, qname, rows, vocabulary, chunk):
    tgo, synth = ops
    qtype, k = QTYPES[qname], 256
    weight = synth.random_packed_weight(qtype, (vocabulary,), k, seed=qtype, scale_range=(1e-3, 3e-2)).cuda()
    targets = torch.from_numpy(np.random.default_rng(rows).integers(0, vocabulary, size=rows)).cuda()
    targets[0], targets[-1] = vocabulary - 1, -100
    hidden = random_bf16((rows, k), seed=7).requires_grad_(True)
    loss = tgo.chunked_lm_head_loss(hidden, weight, targets, qtype, vocabulary, chunk_rows=chunk)
    loss.backward()
    plain = random_bf16((rows, k), seed=7)
    logits = torch.cat([tgo.mmq(part.clone(), weight, qtype, vocabulary) for part in plain.split(chunk)]).float().requires_grad_(True)
    reference = torch.nn.functional.cross_entropy(logits, targets, ignore_index=-100)
    reference.backward()
    expected = torch.ops.torch_ggml_ops.mmq_grad_input.default(logits.grad.bfloat16(), weight, qtype, k)
    torch.testing.assert_close(loss, reference, rtol=1e-5, atol=1e-6)
    assert nrmse(f32(hidden.grad), f32(expected)) < 5e-3
    assert not f32(hidden.grad)[-1].any()
    targets[1] = vocabulary   # neither a column nor ignored
    assert torch.isnan(tgo.chunked_lm_head_loss(hidden.detach(), weight, targets, qtype, vocabulary, chunk_rows=chunk))


@pytest.mark.parametrize("rows", (5, 40))
@pytest.mark.parametrize("columns", ({}, {8192: "nan"}, {8192: "-inf"}, {8192: "nan", 8193: "-inf"}, {8192: "+inf"}, {3: "-inf", 8193: "nan"}))
def test_loss_of_logits_that_are_not_finite(ops, columns, rows):
    """The second span of the vocabulary holds two columns: a NaN there is the row's loss also when nothing finite stands
    beside it, and a span of -inf adds nothing."""
    tgo, synth = ops
    qtype, k, vocabulary = QTYPES["Q4_K"], 256, 8194
    packed = synth.random_packed_weight(qtype, (vocabulary,), k, seed=1, scale_range=(1e-3, 3e-2))
    if columns:
        for column in (8192, 8193):
            columns = {column: next(iter(columns.values())), **columns}
    for column, kind in columns.items():
        # a block of one scale and no minimum: every weight is d * 9 * 1, so that logits are d * 9 * sum(x)
        block = packed.reshape(vocabulary, -1)[column]
        block[:] = torch.tensor([0, 0, 0, 0] + [9] * 4 + [0] * 4 + [9] * 4 + [17] * 128, dtype=torch.uint8)
        block[:2] = torch.tensor({"nan": [0, 0x7E], "-inf": [0, 0x7C], "+inf": [0, 0xFC]}[kind], dtype=torch.uint8)
    weight = packed.cuda()
    hidden = -random_bf16((rows, k), seed=2).abs()   # (a negative sum)
    targets = torch.arange(rows, device="cuda") + 10
    logits = tgo.mmq(hidden, weight, qtype, vocabulary)
    for column, kind in columns.items():
        # (the matrix-core kernels of larger calls make a NaN of an infinite scale, which is the case of the loss then)
        expected = torch.full((rows,), float(kind) if rows == 5 else float("nan"), device="cuda", dtype=torch.bfloat16)
        torch.testing.assert_close(logits[:, column], expected, equal_nan=True)
    reference = torch.nn.functional.cross_entropy(logits.float(), targets)
    assert reference.isnan() == any(kind != "-inf" or rows != 5 for kind in columns.values())
    for gradient in (False, True):
        loss = tgo.chunked_lm_head_loss(hidden.clone().requires_grad_(gradient), weight, targets, qtype, vocabulary)
        torch.testing.assert_close(loss.detach(), reference, rtol=1e-5, atol=1e-6, equal_nan=True)
