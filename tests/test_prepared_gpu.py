"""GPU parity of the prepared-activation operators (-m gpu): quantize once, several projections.

The reference has no such operator, so the oracle here is the library's own ``mmq`` (which the
other tests pin against the CPU oracle): ``mmq_prepared`` must reproduce it bit for bit, and
``mmq_multi``'s gradient must equal the sum of the projections' ``mmq_grad_input``.

A workspace that is quantized before its weight format is known holds int8 tiles and runs the int8 kernels,
while ``mmq`` by default multiplies fp16 operands for IQ2_S: bit-for-bit equality therefore holds with the
int8 operands forced (and by default for the other formats); under the default the two agree up to fp32 rounding.
"""

import pytest
import torch

from helpers import OPERAND_NOISE, QTYPES, assert_matches_f32_reference, bits, random_bf16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import torch_ggml_ops
    import synth

    assert torch.cuda.is_available()
    return torch_ggml_ops, synth


@pytest.fixture(params=("auto", "int8"))
def operand(request):
    from torch_ggml_ops import _native

    _native.set_forward_operand(request.param)
    yield request.param
    _native.set_forward_operand("auto")


def _assert_same(operand, qname, actual, expected):
    if operand == "int8" or qname != "IQ2_S":
        torch.testing.assert_close(actual, expected, rtol=0, atol=0)
    else:   # one bf16 ulp where the fp32 sums round differently
        torch.testing.assert_close(actual.detach().float(), expected.detach().float(), rtol=2.0**-7,
                                   atol=1e-5 * float(expected.detach().float().abs().max()))


@pytest.mark.parametrize("rows", (1, 5, 77, 300))
def test_prepared_equals_mmq_bit_for_bit(ops, oracle, operand, rows):
    tgo, synth = ops
    k = 1024
    x = random_bf16((rows, k), seed=rows)
    workspace = tgo.quantize_q8_1(x)
    assert workspace.dtype == torch.uint8 and workspace.is_cuda
    for qname, n in (("Q4_K", 96), ("Q6_K", 37), ("IQ2_S", 160), ("Q5_K", 512), ("Q3_K", 64)):
        qtype = QTYPES[qname]
        host = synth.random_packed_weight(qtype, (n,), k, seed=700 + qtype)
        weight = host.cuda()
        prepared = tgo.mmq_prepared(workspace, weight, rows, k, qtype, n)
        _assert_same(operand, qname, prepared, tgo.mmq(x, weight, qtype, n))
        assert_matches_f32_reference(prepared, oracle.mmq_forward(qtype, bits(x), host.numpy(), n, k))


def test_multi_projection_forward_and_gradient(ops, operand):
    tgo, synth = ops
    k, shapes = 512, (("Q4_K", 256), ("Q5_K", 64), ("Q6_K", 64))
    weights = [synth.random_packed_weight(QTYPES[q], (n,), k, seed=800 + i).cuda() for i, (q, n) in enumerate(shapes)]
    qtypes = [QTYPES[q] for q, _ in shapes]
    widths = [n for _, n in shapes]
    x = random_bf16((3, 40, k), seed=31).requires_grad_(True)
    outputs = tgo.mmq_multi(x, weights, qtypes, widths)
    grads = [random_bf16((3, 40, n), seed=40 + i) for i, n in enumerate(widths)]
    torch.autograd.backward(outputs, grads)

    y = x.detach().clone().requires_grad_(True)
    separate = [tgo.mmq(y, w, q, n) for w, q, n in zip(weights, qtypes, widths)]
    for fused, plain, (qname, _) in zip(outputs, separate, shapes):
        assert fused.shape == plain.shape
        _assert_same(operand, qname, fused, plain)
    expected = None
    for grad, weight, qtype in zip(grads, weights, qtypes):
        term = torch.ops.torch_ggml_ops.mmq_grad_input.default(grad, weight, qtype, k)
        expected = term if expected is None else expected + term
    torch.testing.assert_close(x.grad, expected, rtol=0, atol=0)

    # a projection whose output is unused contributes nothing
    z = x.detach().clone().requires_grad_(True)
    first, _, _ = tgo.mmq_multi(z, weights, qtypes, widths)
    first.backward(grads[0])
    only = torch.ops.torch_ggml_ops.mmq_grad_input.default(grads[0], weights[0], qtypes[0], k)
    torch.testing.assert_close(z.grad, only, rtol=0, atol=0)


@pytest.mark.parametrize("kind", ("int8", "half", "scaled"))
def test_workspace_of_a_named_kind_matches_the_oracle(ops, oracle, kind):
    """A caller may name the operand kind of a workspace: every format's kernel of that kind reads it."""
    tgo, synth = ops
    rows, k = 300, 1024
    x = random_bf16((rows, k), seed=17)
    workspace = tgo.quantize_q8_1(x, operand=kind)
    for qname, n in (("Q4_K", 96), ("Q6_K", 37), ("IQ2_S", 160), ("Q5_K", 512), ("Q3_K", 64)):
        qtype = QTYPES[qname]
        host = synth.random_packed_weight(qtype, (n,), k, seed=900 + qtype)
        prepared = tgo.mmq_prepared(workspace, host.cuda(), rows, k, qtype, n, operand=kind)
        assert_matches_f32_reference(prepared, oracle.mmq_forward(qtype, bits(x), host.numpy(), n, k),
                                     accumulate_noise=OPERAND_NOISE[kind])
    # the same workspace read as another kind: refused on the device, every output NaN
    other = "int8" if kind != "int8" else "scaled"
    weight = synth.random_packed_weight(12, (64,), k, seed=5).cuda()
    assert torch.isnan(tgo.mmq_prepared(workspace, weight, rows, k, 12, 64, operand=other).float()).all()
    with pytest.raises(ValueError, match="operand must be"):
        tgo.quantize_q8_1(x, operand="fp8")


def test_multi_projection_of_a_long_sequence_takes_the_scaled_kernels(ops):
    """q/k/v of 2048 rows fill the chip together: mmq_multi quantizes for, and runs, the scaled kernels, and each
    projection agrees with a separate mmq (scaled or int8 by its own size) within the scaled kind's rounding."""
    from torch_ggml_ops import prepared

    tgo, synth = ops
    rows, k, widths = 2048, 512, (2048, 1024, 1024)
    qtypes = [QTYPES["Q4_K"], QTYPES["Q4_K"], QTYPES["Q6_K"]]
    assert prepared.multi_operand(qtypes, rows, widths) == "scaled"
    assert prepared.multi_operand(qtypes, 40, widths) == "int8"
    assert prepared.multi_operand([QTYPES["IQ2_S"]] * 2, 40, widths[:2]) == "half"
    assert prepared.multi_operand([QTYPES["IQ2_S"], QTYPES["Q4_K"]], 40, widths[:2]) == "int8"
    weights = [synth.random_packed_weight(q, (n,), k, seed=60 + i).cuda() for i, (q, n) in enumerate(zip(qtypes, widths))]
    x = random_bf16((rows, k), seed=9)
    outputs = tgo.mmq_multi(x, weights, qtypes, widths)
    for output, weight, qtype, n in zip(outputs, weights, qtypes, widths):
        plain = tgo.mmq(x, weight, qtype, n).float()
        tolerance = plain.abs() * 2.0**-7 + 2 * OPERAND_NOISE["scaled"] * float(plain.abs().max())
        assert bool(((output.float() - plain).abs() <= tolerance).all())


def test_prepared_rejects_mismatched_workspace(ops):
    tgo, synth = ops
    x = random_bf16((8, 512), seed=1)
    workspace = tgo.quantize_q8_1(x)
    weight = synth.random_packed_weight(12, (32,), 512, seed=2).cuda()
    with pytest.raises(RuntimeError, match="workspace holds"):
        tgo.mmq_prepared(workspace, weight, 64, 512, 12, 32)
    with pytest.raises(RuntimeError, match="packed_weight has"):
        tgo.mmq_prepared(workspace, weight, 8, 512, 13, 32)
    with pytest.raises(RuntimeError, match="multiple of 256"):
        tgo.quantize_q8_1(random_bf16((4, 100), seed=3))


@pytest.mark.parametrize("qname", tuple(QTYPES))
@pytest.mark.parametrize("rows,n,k", [(33, 4096, 1024), (48, 2048, 2304), (64, 16400, 768), (61, 2064, 4096), (128, 2048, 2048)])
def test_rows_beyond_the_decode_regime_equal_mmq_bit_for_bit(ops, oracle, qname, rows, n, k):
    """Matrices of four million weights, which ``mmq`` gives to the 16-row decode kernel for up to 128 rows: a workspace in either
    exact tile layout, and ``mmq_multi``, give the same bits (the kernel's sums do not depend on how its activations are laid
    out), also a key and value of one shape and a projection that takes the matrix-core kernels."""
    from torch_ggml_ops import _native, prepared

    tgo, synth = ops
    qtype = QTYPES[qname]
    assert _native.forward_kernel_for(qtype, rows, k, n) == "tiles"
    host = synth.random_packed_weight(qtype, (n,), k, seed=qtype + rows)
    weight = host.cuda()
    x = random_bf16((rows, k), seed=rows)
    expected = tgo.mmq(x, weight, qtype, n)
    assert_matches_f32_reference(expected, oracle.mmq_forward(qtype, bits(x), host.numpy(), n, k))
    for kind in ("int8", "half"):
        actual = tgo.mmq_prepared(tgo.quantize_q8_1(x, kind), weight, rows, k, qtype, n, kind)
        torch.testing.assert_close(actual, expected, rtol=0, atol=0)
    other = synth.random_packed_weight(qtype, (n,), k, seed=1).cuda()
    small = synth.random_packed_weight(qtype, (n // 16 + 1,), k, seed=2).cuda()
    widths = (n, n, n // 16 + 1)
    assert _native.forward_kernel_for(qtype, rows, k, widths[2]) == "mfma"
    if prepared.multi_operand([qtype] * 3, rows, widths) != "scaled":
        outputs = tgo.mmq_multi(x, (weight, other, small), [qtype] * 3, widths)
        for output, w, width in zip(outputs, (weight, other, small), widths):
            torch.testing.assert_close(output, tgo.mmq(x, w, qtype, width), rtol=0, atol=0)


def test_another_layout_than_the_workspaces_is_nan_on_the_decode_kernel_too(ops):
    tgo, synth = ops
    rows, n, k = 40, 4096, 1024
    weight = synth.random_packed_weight(12, (n,), k, seed=3).cuda()
    workspace = tgo.quantize_q8_1(random_bf16((rows, k), seed=4), operand="half")
    assert torch.isnan(tgo.mmq_prepared(workspace, weight, rows, k, 12, n, operand="int8").float()).all()


@pytest.mark.parametrize("call", ("prepared", "multi", "int8", "half"))
def test_calls_that_do_not_unpack_their_weights_have_no_scratch_for_them(ops, call):
    """Two bytes per weight, where ``mmq`` with scaled operands has them."""
    tgo, synth = ops
    from torch_ggml_ops import _native

    qtype, rows, k, n = 12, 4096, 4096, 4096
    unpacked = _native.lib.tgo_forward_scratch_bytes_as(rows, k, n, qtype, _native.OPERANDS["scaled"])
    assert unpacked >= 2 * n * k
    packed = synth.random_packed_weight(qtype, (n,), k, seed=1).cuda()
    other = synth.random_packed_weight(14, (n,), k, seed=2).cuda()   # (of another format: not one product)
    x = random_bf16((rows, k), seed=3)
    workspace = tgo.quantize_q8_1(x, "scaled")
    try:
        if call in ("int8", "half"):
            _native.set_forward_operand(call)
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        if call == "prepared":
            outputs = [tgo.mmq_prepared(workspace, packed, rows, k, qtype, n, "scaled")]
        elif call == "multi":
            outputs = tgo.mmq_multi(x, [packed, other], [qtype, 14], [n, n])
        else:
            outputs = [tgo.mmq(x, packed, qtype, n)]
        taken = torch.cuda.max_memory_allocated() - before
    finally:
        _native.set_forward_operand("auto")
    kept = sum(o.numel() * 2 for o in outputs) + (0 if call == "prepared" else workspace.numel())
    assert taken < kept + unpacked // 4


def test_scratch_that_is_too_small_is_done_without(ops):
    """A call whose scratch was sized under another setting: the same bits as without scratch, and nothing written beyond it."""
    _, synth = ops
    from torch_ggml_ops import _native

    qtype, rows, k, n, lib = 12, 2048, 2048, 2048, _native.lib
    needed = lib.tgo_forward_scratch_bytes_as(rows, k, n, qtype, _native.OPERANDS["scaled"])
    assert needed > 0
    packed = synth.random_packed_weight(qtype, (n,), k, seed=1).cuda()
    x = random_bf16((rows, k), seed=3)
    workspace = torch.empty(lib.tgo_q8_workspace_bytes(rows, k), dtype=torch.uint8, device="cuda")
    scratch = torch.full((needed,), 0x5A, dtype=torch.uint8, device="cuda")
    outputs = []
    for size in (0, needed - 1, needed):
        assert bool((scratch == 0x5A).all())
        output = torch.empty((rows, n), dtype=torch.bfloat16, device="cuda")
        _native.check(lib.tgo_mmq_forward_sized(x.data_ptr(), packed.data_ptr(), output.data_ptr(), workspace.data_ptr(), scratch.data_ptr(), size,
                                                rows, k, n, qtype, _native.stream_of(x.device)))
        outputs.append(output)
    assert torch.equal(outputs[0], outputs[1]) and torch.equal(outputs[0], outputs[2])
    assert not bool((scratch == 0x5A).all())
