"""tgo_forward_kernel_for names the kernels that ran (-m gpu): the library's own launch brackets tell the decode kernels from the
matrix-core ones."""

import pytest
import torch

from helpers import QTYPES, random_bf16

pytestmark = pytest.mark.gpu


def _ran(native, call):
    native.lib.tgo_profile_enable(1)
    try:
        call()
        decode, matrix = native.profile_read("forward_gemv")[1], native.profile_read("forward")[1]
    finally:
        native.lib.tgo_profile_enable(0)
    assert (decode > 0) != (matrix > 0)
    return "decode" if decode > 0 else "mfma"


@pytest.mark.parametrize("qname", tuple(QTYPES))
def test_dense_and_grouped(qname):
    import synth
    import torch_ggml_ops as tgo
    from torch_ggml_ops import _native

    qtype = QTYPES[qname]
    names = set()
    for rows, n, k in ((4, 2048, 2048), (32, 2048, 2048), (33, 2048, 2048), (128, 2048, 2048), (129, 2048, 2048), (64, 2050, 2048), (64, 512, 2048)):
        weight = synth.random_packed_weight(qtype, (n,), k, seed=1).cuda()
        x = random_bf16((rows, k), seed=rows)
        name = _native.forward_kernel_for(qtype, rows, k, n)
        names.add(name)
        assert _ran(_native, lambda: tgo.mmq(x, weight, qtype, n)) == ("mfma" if name == "mfma" else "decode"), (rows, n, k)
    experts, n, k = 16, 1024, 512
    weight = synth.random_packed_weight(qtype, (experts, n), k, seed=2).cuda()
    for rows in (8, 16, 5 * experts, 8 * experts, 40 * experts):
        ends = torch.linspace(0, rows, experts + 1, device="cuda")[1:].round().to(torch.int32)
        x = random_bf16((rows, k), seed=rows)
        for pair in (False, True):
            name = _native.forward_kernel_for(qtype, rows, k, n, experts, 2 if pair else 1)
            names.add(name)
            operands = (torch.arange(experts, device="cuda"), ends, qtype, n)
            call = (lambda: tgo.grouped_mmq_pair(x, weight, weight, *operands)) if pair else (lambda: tgo.grouped_mmq(x, weight, *operands))
            assert _ran(_native, call) == ("mfma" if name == "mfma" else "decode"), (rows, pair)
    assert {"tiles", "mfma"} <= names
