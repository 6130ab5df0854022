"""GPU parity of the decode-regime kernel for tasks of several rows against the CPU oracle (-m gpu): its edges are the
16 rows of a task, the 16 weight rows of a tile (a last workgroup with tiles missing, one and several waves per
tile), the two, four or fewer shares of K, and weight blocks at every address modulo 16 up to the tensor's last."""

import numpy as np
import pytest
import torch

from helpers import QTYPES, assert_matches_f32_reference, bits, random_bf16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import torch_ggml_ops
    import synth

    assert torch.cuda.is_available()
    return torch_ggml_ops, synth


@pytest.mark.parametrize("qname", tuple(QTYPES))
@pytest.mark.parametrize("rows,n,k", [(17, 16400, 256), (32, 5472, 768), (5, 3280, 1280), (20, 1840, 2304), (9, 2064, 16384)])
def test_dense(ops, oracle, qname, rows, n, k):
    tgo, synth = ops
    qtype = QTYPES[qname]
    host = synth.random_packed_weight(qtype, (n,), k, seed=700 + qtype + rows)
    x = random_bf16((rows, k), seed=rows)
    assert_matches_f32_reference(tgo.mmq(x, host.cuda(), qtype, n), oracle.mmq_forward(qtype, bits(x), host.numpy(), n, k))


@pytest.mark.parametrize("qname", tuple(QTYPES))
@pytest.mark.parametrize("n,k", [(2048, 512), (816, 256), (208, 1024), (96, 2304)])
def test_grouped(ops, oracle, qname, n, k):
    """Groups of 1 to 33 rows (up to three tasks), empty ones, an expert that does not exist."""
    tgo, synth = ops
    qtype, experts = QTYPES[qname], 24
    host = [synth.random_packed_weight(qtype, (experts, n), k, seed=seed + qtype) for seed in (800, 900)]
    sizes = [1, 16, 0, 2, 33, 0, 5, 1, 17, 3, 0, 1, 1, 4, 1, 2, 0, 1, 1, 0, 3]
    chosen = np.random.default_rng(5).permutation(experts)[: len(sizes)].tolist()
    chosen[3] = experts
    offsets = np.cumsum(sizes).tolist()
    x = random_bf16((offsets[-1], k), seed=31)
    indices = torch.tensor(chosen, dtype=torch.int64, device="cuda")
    ends = torch.tensor(offsets, dtype=torch.int32, device="cuda")
    outputs = tgo.grouped_mmq_pair(x, host[0].cuda(), host[1].cuda(), indices, ends, qtype, n)
    exact = [oracle.grouped(oracle.mmq_forward, qtype, bits(x), h.numpy(), chosen, offsets, n, k, n) for h in host]
    covered = ~np.isnan(exact[0][:, 0])
    assert covered.sum() == offsets[-1] - 2
    on_device = torch.from_numpy(covered).cuda()
    for actual, expected in zip(outputs, exact):
        assert_matches_f32_reference(actual[on_device], expected[covered])
    activated = tgo.grouped_mmq_swiglu(x, host[0].cuda(), host[1].cuda(), indices, ends, qtype, n)
    gate, up = (o.float() for o in outputs)
    expected = (torch.nn.functional.silu(gate) * up)[on_device]
    assert ((activated.float()[on_device] - expected).abs() <= 2.0**-7 * expected.abs() + 1e-6).all()


@pytest.mark.parametrize("qname", tuple(QTYPES))
@pytest.mark.parametrize("n,sizes", [(512, [1, 15, 16, 17, 33, 5, 0, 2] * 2), (2048, [40, 3, 1, 18])])
def test_grouped_calls_of_a_few_rows_per_group(oracle, qname, n, sizes):
    """Beyond the decode regime (more than four rows per group on average): groups of one to three tasks of 16 rows, none, and a list
    of four groups whose K and columns make up the four million weights; one projection and a pair."""
    import synth
    import torch_ggml_ops as tgo

    qtype, k = QTYPES[qname], 512
    experts = list(range(len(sizes)))[::-1]
    offsets = np.cumsum(sizes).tolist()
    assert 4 * len(sizes) < offsets[-1] <= 16 * len(sizes)
    metadata = (torch.tensor(experts, device="cuda"), torch.tensor(offsets, device="cuda", dtype=torch.int32))
    hosts = [synth.random_packed_weight(qtype, (len(sizes), n), k, seed=qtype + i) for i in range(2)]
    weights = [host.cuda() for host in hosts]
    x = random_bf16((offsets[-1], k), seed=n)
    expected = [oracle.grouped(oracle.mmq_forward, qtype, bits(x), host.numpy(), experts, offsets, n, k, n) for host in hosts]
    assert_matches_f32_reference(tgo.grouped_mmq(x, weights[0], *metadata, qtype, n), expected[0])
    first, second = tgo.grouped_mmq_pair(x, *weights, *metadata, qtype, n)
    assert_matches_f32_reference(first, expected[0])
    assert_matches_f32_reference(second, expected[1])


@pytest.mark.parametrize("qname", tuple(QTYPES))
@pytest.mark.parametrize("rows,n,k", [(33, 4096, 1024), (64, 16400, 768), (81, 2064, 4096), (128, 5120, 1024), (129, 5120, 1024)])
def test_dense_beyond_the_decode_regime(oracle, qname, rows, n, k):
    """Three to eight tasks of 16 rows, the last one not full, and one row beyond the line."""
    import synth
    import torch_ggml_ops as tgo

    qtype = QTYPES[qname]
    host = synth.random_packed_weight(qtype, (n,), k, seed=qtype + rows)
    x = random_bf16((rows, k), seed=rows)
    assert_matches_f32_reference(tgo.mmq(x, host.cuda(), qtype, n), oracle.mmq_forward(qtype, bits(x), host.numpy(), n, k))


@pytest.mark.parametrize("qname", tuple(QTYPES))
@pytest.mark.parametrize("rows,n,k,taken", [(17, 256, 512, True), (31, 16, 8192, True), (32, 1040, 2304, True), (24, 2064, 1024, True), (33, 256, 512, False),
                                            (20, 480, 256, False), (32, 520, 1024, False)])
def test_dense_decode_on_few_weights(oracle, qname, rows, n, k, taken):
    """From 2^17 to below 2^22 weights: one tile of weight rows, a last workgroup that lacks tiles, a task of one row less than two, the most rows
    and one more, too few weights, a matrix that is not made of whole tiles."""
    import synth
    import torch_ggml_ops as tgo
    from torch_ggml_ops import _native

    qtype = QTYPES[qname]
    assert (_native.forward_kernel_for(qtype, rows, k, n) == "tiles") == taken
    host = synth.random_packed_weight(qtype, (n,), k, seed=qtype + rows)
    x = random_bf16((rows, k), seed=rows)
    assert_matches_f32_reference(tgo.mmq(x, host.cuda(), qtype, n), oracle.mmq_forward(qtype, bits(x), host.numpy(), n, k))


@pytest.mark.parametrize("qname", tuple(QTYPES))
def test_grouped_and_dense_calls_on_this_kernel_have_the_same_bits(qname):
    """Groups of 1 to 50 rows of a grouped call that averages eleven, and a dense call on each of them: where both run on this kernel, the
    same bits."""
    import synth
    import torch_ggml_ops as tgo
    from torch_ggml_ops import _native

    qtype, n, k = QTYPES[qname], 2048, 2048
    sizes = [50, 1, 40, 3, 16, 17, 1, 2, 1, 33, 1, 1, 1, 1, 2, 5]
    experts = len(sizes)
    ends = np.cumsum(sizes).tolist()
    weight = synth.random_packed_weight(qtype, (experts, n), k, seed=qtype).cuda()
    x = random_bf16((ends[-1], k), seed=6)
    assert _native.forward_kernel_for(qtype, ends[-1], k, n, experts) == "tiles" and ends[-1] > 4 * experts
    output = tgo.grouped_mmq(x, weight, torch.arange(experts, device="cuda"), torch.tensor(ends, device="cuda", dtype=torch.int32), qtype, n)
    compared = 0
    for expert, (begin, end) in enumerate(zip([0] + ends, ends)):
        if _native.forward_kernel_for(qtype, end - begin, k, n) == "tiles":
            dense = tgo.mmq(x[begin:end].clone(), weight[expert].clone(), qtype, n)
            torch.testing.assert_close(output[begin:end], dense, rtol=0, atol=0)
            compared += 1
    assert compared >= 4
