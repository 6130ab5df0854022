"""Dense products whose weights are unpacked once per call (-m gpu) against float64 products of the oracle's weights: every tile shape
of the product, rows that end inside a tile, whole rounds of tiles with rows behind them, cotangents that are read as they stand and
cotangents that are packed (columns that are no multiple of 32), several projections as one reduction."""

import ctypes

import numpy as np
import pytest
import torch

from helpers import QTYPES, assert_matches_f32_reference, random_bf16

pytestmark = pytest.mark.gpu


def _weights(oracle, qtype, widths, k):
    """Packed weights, and the oracle's bf16 values of them as float64."""
    import synth

    host = [synth.random_packed_weight(q, (n,), k, seed=q + n + i) for i, (q, n) in enumerate(zip(qtype, widths))]
    plain = [torch.from_numpy(oracle.bf16_to_f32(oracle.dequant_bf16(q, h.numpy(), k)).astype(np.float64)).cuda() for q, h in zip(qtype, host)]
    return [h.cuda() for h in host], plain


def _unpacks_gradient(rows, widths, k):
    from torch_ggml_ops import _native

    return _native.lib.tgo_multi_grad_workspace_bytes(len(widths), (ctypes.c_int64 * len(widths))(*widths), rows, k) > 0


# (rows, weight rows, K): 128 x 128 tiles, one row behind a tile and one short of it; odd reductions, which pack; 128 x 256 tiles; whole rounds of
# 256 x 256 tiles and rows behind them, packed and not; more than eight row tiles, which are dealt out in bands
GRADIENTS = [(257, 640, 768), (255, 623, 2304), (1731, 1859, 512), (4000, 1056, 2048), (4200, 544, 4096), (4133, 521, 4096), (9000, 96, 512)]


@pytest.mark.parametrize("qname", tuple(QTYPES))
@pytest.mark.parametrize("rows,n,k", GRADIENTS)
def test_gradient(oracle, qname, rows, n, k):
    assert _unpacks_gradient(rows, [n], k)
    (packed,), (plain,) = _weights(oracle, [QTYPES[qname]], [n], k)
    grad = random_bf16((rows, n), seed=rows)
    actual = torch.ops.torch_ggml_ops.mmq_grad_input.default(grad, packed, QTYPES[qname], k)
    assert_matches_f32_reference(actual, (grad.double() @ plain).cpu().numpy(), accumulate_noise=1e-5)
    one_hot = torch.zeros_like(grad)
    one_hot[rows - 1, n - 1] = 1
    picked = torch.ops.torch_ggml_ops.mmq_grad_input.default(one_hot, packed, QTYPES[qname], k)
    assert torch.equal(picked[rows - 1].double(), plain[n - 1]) and not picked[: rows - 1].any()


@pytest.mark.parametrize("widths", [(2048, 512, 512), (1000, 250, 250), (608, 96), (512, 512, 512, 512)])
def test_gradient_of_several_projections(oracle, widths):
    """Formats of their own, widths whose 64-row steps are filled up, and the sum rounded once."""
    import torch_ggml_ops as tgo

    rows, k = 700, 2048
    assert _unpacks_gradient(rows, widths, k)
    qtypes = [QTYPES[q] for q in ("Q4_K", "Q6_K", "IQ2_S", "Q3_K")][: len(widths)]
    packed, plain = _weights(oracle, qtypes, widths, k)
    x = random_bf16((rows, k), seed=1).requires_grad_()
    grads = [random_bf16((rows, n), seed=5 + i) for i, n in enumerate(widths)]
    outputs = tgo.mmq_multi(x, packed, qtypes, widths)
    (grad,) = torch.autograd.grad(outputs, x, grads)
    expected = sum(g.double() @ p for g, p in zip(grads, plain))
    assert_matches_f32_reference(grad, expected.cpu().numpy(), accumulate_noise=1e-5)
