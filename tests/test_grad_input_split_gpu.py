"""GPU parity of the role-split grad-input kernel against the CPU oracle (-m gpu), every format: rows on both sides of its
256-row and 32-row tiles, reductions that end inside a 64-row step, an odd number of super-blocks of K, whole reductions,
several ranges of one, and ranges of unequal length."""

import numpy as np
import pytest
import torch

from helpers import QTYPES, assert_matches_f32_reference, bits, random_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qname", tuple(QTYPES))
@pytest.mark.parametrize(
    "rows,n,k", [(1, 40, 256), (33, 130, 768), (256, 1003, 512), (257, 2111, 1280), (70, 4096, 256), (2304, 192, 1280), (1000, 2049, 8192)]
)
def test_dense(oracle, qname, rows, n, k):
    import synth
    import torch_ggml_ops  # noqa: F401

    qtype = QTYPES[qname]
    host = synth.random_packed_weight(qtype, (n,), k, seed=qtype + rows)
    grad = random_bf16((rows, n), seed=rows)
    actual = torch.ops.torch_ggml_ops.mmq_grad_input.default(grad, host.cuda(), qtype, k)
    # (the largest calls: the first rows, some in the middle of the second tile, and the last)
    picked = np.arange(rows) if rows * n * k < 2**29 else np.r_[0:8, rows // 2 : rows // 2 + 8, rows - 8 : rows]
    expected = oracle.grad_input(qtype, bits(grad)[picked], host.numpy(), n, k)
    assert_matches_f32_reference(actual[torch.from_numpy(picked).cuda()], expected, accumulate_noise=1e-5)
