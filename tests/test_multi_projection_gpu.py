"""Projections of one shape and format inside ``mmq_multi`` run as pairs (-m gpu): the bits of ``mmq_prepared`` forward, and a
gradient that is the fp32 sum rounded once."""

import numpy as np
import pytest
import torch

from helpers import QTYPES, assert_matches_f32_reference, bits, random_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qname", tuple(QTYPES))
@pytest.mark.parametrize("rows,n,kv,k", [(40, 96, 40, 512), (300, 2000, 500, 1024), (2048, 1024, 256, 512)])
def test_key_and_value(oracle, qname, rows, n, kv, k):
    import synth
    import torch_ggml_ops as tgo
    from torch_ggml_ops import prepared

    qtype, widths = QTYPES[qname], (n, kv, kv)
    host = [synth.random_packed_weight(qtype, (w,), k, seed=10 + i + qtype) for i, w in enumerate(widths)]
    device = [h.cuda() for h in host]
    x = random_bf16((rows, k), seed=1).requires_grad_()
    outputs = tgo.mmq_multi(x, device, [qtype] * 3, widths)
    operand = prepared.multi_operand([qtype] * 3, rows, widths)
    workspace = tgo.quantize_q8_1(x.detach(), operand)
    for output, weight, width in zip(outputs, device, widths):
        expected = tgo.mmq_prepared(workspace, weight, rows, k, qtype, width, operand)
        torch.testing.assert_close(output.detach(), expected, rtol=0, atol=0)
    grads = [random_bf16((rows, w), seed=5 + i) for i, w in enumerate(widths)]
    (grad,) = torch.autograd.grad(outputs[1:], x, grads[1:])
    picked = np.r_[0:20, rows - 20 : rows]
    expected = sum(oracle.grad_input(qtype, bits(g)[picked], h.numpy(), kv, k).astype(np.float64) for g, h in zip(grads[1:], host[1:]))
    assert_matches_f32_reference(grad[torch.from_numpy(picked).cuda()], expected, accumulate_noise=1e-5)
