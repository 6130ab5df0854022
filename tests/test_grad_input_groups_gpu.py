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


@pytest.mark.parametrize("qname", ("Q4_K", "Q5_K", "IQ2_S"))
@pytest.mark.parametrize("short", (1, 33, 64, 65))
def test_groups_whose_cotangent_is_longer_than_32_bits_reach(oracle, qname, short):
    """Four GiB of packed cotangent in front of the last groups, and several steps of the reduction."""
    import synth
    import torch_ggml_ops as tgo  # noqa: F401

    qtype, n, k, experts = QTYPES[qname], 4096, 256, 3
    sizes = [2**31 // n, 7, short]
    ends = np.cumsum(sizes).tolist()
    host = synth.random_packed_weight(qtype, (experts, n), k, seed=qtype + short)
    grad = torch.empty((ends[-1], n), dtype=torch.bfloat16, device="cuda")
    generator = torch.Generator(device="cuda").manual_seed(short)
    for first in range(0, ends[-1], 2**16):
        grad[first : first + 2**16].normal_(generator=generator)
    metadata = (torch.arange(experts, device="cuda"), torch.tensor(ends, device="cuda", dtype=torch.int32))
    actual = torch.ops.torch_ggml_ops.grouped_mmq_grad_input.default(grad, host.cuda(), *metadata, qtype, k)
    picked = np.r_[0:4, ends[0] - 4 : ends[-1]]
    expert = np.searchsorted(ends, picked, side="right")
    plain = [oracle.bf16_to_f32(oracle.dequant_bf16(qtype, host[e].numpy(), k)).astype(np.float64) for e in range(experts)]
    values = grad[torch.from_numpy(picked).cuda()].double().cpu().numpy()
    expected = np.stack([row @ plain[e] for row, e in zip(values, expert)])
    assert_matches_f32_reference(actual[torch.from_numpy(picked).cuda()], expected, accumulate_noise=1e-5)


@pytest.mark.parametrize("qname", ("Q4_K", "Q6_K"))
def test_groups_of_more_weight_rows_than_the_short_kernel_reaches(oracle, qname):
    """22.4 million weight rows, of which a cotangent that is mostly zeros picks a few, the first and the last ones among them."""
    import synth
    import torch_ggml_ops as tgo  # noqa: F401

    qtype, n, k, sizes = QTYPES[qname], 22_400_000, 256, [3, 65]
    weight = synth.random_packed_weight(qtype, (2, n), k, seed=qtype, device="cuda")
    ends = np.cumsum(sizes).tolist()
    grad = torch.zeros((ends[-1], n), dtype=torch.bfloat16, device="cuda")
    columns = torch.tensor([0, 63, 64, 1 << 23, n // 2 + 1, n - 65, n - 1], device="cuda")
    grad[:, columns] = random_bf16((ends[-1], columns.numel()), seed=qtype)
    metadata = (torch.arange(2, device="cuda"), torch.tensor(ends, device="cuda", dtype=torch.int32))
    actual = torch.ops.torch_ggml_ops.grouped_mmq_grad_input.default(grad, weight, *metadata, qtype, k)
    plain = [oracle.bf16_to_f32(oracle.dequant_bf16(qtype, weight[e, columns].cpu().numpy(), k)).astype(np.float64) for e in range(2)]
    values = grad[:, columns].double().cpu().numpy()
    expected = np.concatenate([values[: sizes[0]] @ plain[0], values[sizes[0] :] @ plain[1]])
    assert_matches_f32_reference(actual, expected, accumulate_noise=1e-6)
