"""GPU parity of dense forward calls whose K is cut into ranges against the CPU oracle (-m gpu): both exact operand kinds, every
format, rows and columns that end inside a tile, the narrow and the full row tiles, ranges of unequal length."""

import numpy as np
import pytest
import torch

from helpers import QTYPES, assert_matches_f32_reference, bits, random_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qname", tuple(QTYPES))
@pytest.mark.parametrize("operand", ("int8", "half"))
@pytest.mark.parametrize("rows,n,k", [(33, 4097, 1024), (70, 2003, 2304), (130, 1000, 4352), (600, 1100, 4096)])
def test_dense(oracle, qname, operand, rows, n, k):
    import synth
    import torch_ggml_ops as tgo
    from torch_ggml_ops import _native

    qtype = QTYPES[qname]
    host = synth.random_packed_weight(qtype, (n,), k, seed=qtype + rows)
    x = random_bf16((rows, k), seed=rows)
    assert _native.lib.tgo_forward_scratch_bytes(rows, k, n, qtype) > 0
    picked = np.arange(rows) if rows < 200 else np.r_[0:8, 250:262, rows - 8 : rows]
    workspace = tgo.quantize_q8_1(x, operand)
    actual = tgo.mmq_prepared(workspace, host.cuda(), rows, k, qtype, n, operand)
    expected = oracle.mmq_forward(qtype, bits(x)[picked], host.numpy(), n, k)
    assert_matches_f32_reference(actual[torch.from_numpy(picked).cuda()], expected)
    if operand == _native.forward_operand_for(qtype, rows, n):
        torch.testing.assert_close(tgo.mmq(x, host.cuda(), qtype, n), actual, rtol=0, atol=0)
