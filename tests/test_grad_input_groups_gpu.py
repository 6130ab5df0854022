"""Grouped grad-input of short groups (at most 64 rows, a kernel of their own) and longer ones against float64 products of the oracle's weights (-m gpu):
one row to a row beyond the line, one and two row tiles; weight rows that leave a step of 64 or a wave's 16 of it incomplete, one step and several;
blocks at every even address modulo 16, experts whose bytes are no whole number of 16; one projection and a pair."""

import numpy as np
import pytest
import torch

from helpers import QTYPES, assert_matches_f32_reference, bits, random_bf16

pytestmark = pytest.mark.gpu

SIZES = [1, 31, 32, 0, 33, 63, 64, 65, 7, 300]


@pytest.mark.parametrize("qname", tuple(QTYPES))
@pytest.mark.parametrize("n,k", [(5, 256), (37, 768), (64, 256), (79, 512), (130, 256), (321, 768)])
def test_groups(oracle, qname, n, k):
    import synth
    import torch_ggml_ops as tgo  # noqa: F401

    qtype, experts = QTYPES[qname], len(SIZES)
    hosts = [synth.random_packed_weight(qtype, (experts, n), k, seed=40 + qtype + i) for i in range(2)]
    order, ends = list(range(experts))[::-1], np.cumsum(SIZES).tolist()
    metadata = (torch.tensor(order, device="cuda"), torch.tensor(ends, device="cuda", dtype=torch.int32))
    grads = [random_bf16((ends[-1], n), seed=n + i) for i in range(2)]
    expected = [oracle.grouped(oracle.grad_input, qtype, bits(g), h.numpy(), order, ends, n, k, k) for g, h in zip(grads, hosts)]
    weights = [h.cuda() for h in hosts]
    single = torch.ops.torch_ggml_ops.grouped_mmq_grad_input.default(grads[0], weights[0], *metadata, qtype, k)
    assert_matches_f32_reference(single, expected[0], accumulate_noise=2e-6)
    pair = torch.ops.torch_ggml_ops.grouped_mmq_pair_grad_input.default(*grads, *weights, *metadata, qtype, k)
    both = (expected[0].astype(np.float64) + expected[1]).astype(np.float32)
    assert_matches_f32_reference(pair, both, accumulate_noise=2e-6)
