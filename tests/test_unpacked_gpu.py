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
GRADIENTS = [(257, 640, 768), (255, 623, 2304), (1731, 1859, 512), (4000, 1056, 2048), (4200, 1568, 4096), (4133, 1569, 4096), (9000, 96, 512)]


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


@pytest.mark.parametrize("qname", ("Q4_K", "IQ2_S"))
def test_gradient_workspaces(qname):
    """One buffer for calls on either side of the rule: nothing that an earlier call left there is read, and nothing is written beyond the bytes that a
    call asks for, with cotangents that are read as they stand and cotangents that are packed."""
    import synth
    import torch_ggml_ops  # noqa: F401
    from torch_ggml_ops import _native

    qtype, lib, k = QTYPES[qname], _native.lib, 2048
    buffer = torch.full((1 << 26,), 0xFF, dtype=torch.uint8, device="cuda")
    stream = _native.stream_of(buffer.device)
    unpack = []
    for rows, n in ((4000, 1056), (40, 1056), (4133, 1569), (300, 640), (4000, 1056), (64, 1569), (4133, 1569)):
        size = lib.tgo_dense_grad_workspace_bytes(rows, n, k, qtype)
        unpack.append(_unpacks_gradient(rows, [n], k))
        if unpack[-1]:
            assert size == 2 * n * k if n % 32 == 0 else size >= 2 * n * (k + rows)
        packed = synth.random_packed_weight(qtype, (n,), k, seed=qtype + n).cuda()
        grad = random_bf16((rows, n), seed=rows)
        expected = torch.ops.torch_ggml_ops.mmq_grad_input.default(grad, packed, qtype, k)
        actual = torch.empty((rows, k), dtype=torch.bfloat16, device="cuda")
        buffer[size:] = 0xA5
        _native.check(lib.tgo_mmq_grad_input(grad.data_ptr(), packed.data_ptr(), actual.data_ptr(), buffer.data_ptr(), rows, n, k, qtype, stream))
        assert torch.equal(actual, expected) and bool((buffer[size:] == 0xA5).all())
    assert unpack.count(True) >= 4 and not unpack[1] and not unpack[5]


# (rows, columns, K): 128 x 128 and 128 x 256 tiles; an odd number of super-blocks and with it of the minima's steps (K = 768, 1280); columns that end
# inside a tile; rows of 16-byte units and not (Q3_K, Q6_K and IQ2_S of K = 768 and an odd number of columns); 256 x 256 tiles, whole rounds of them
# and rows behind those.  Every call here has to unpack its weights: of short reductions Q4_K and Q5_K do not.
FORWARDS = [(2000, 2048, 2048), (1000, 5003, 1280), (9000, 520, 512), (4097, 4096, 1280), (8300, 2041, 1280), (2600, 5000, 1280)]
SHORT_FORWARDS = [(545, 6017, 768), (8200, 769, 768), (4097, 4096, 1024)]


@pytest.mark.parametrize(
    "qname,rows,n,k", [(q, *f) for q in QTYPES for f in FORWARDS + (SHORT_FORWARDS if q in ("Q3_K", "Q6_K", "IQ2_S") else [])]
)
def test_forward_has_the_bits_of_the_scaled_kernel(qname, rows, n, k):
    """The same operands in the same order: a call without scratch, which the scaled kernel takes, gives the same bits.  Super-blocks far below
    their row's largest one, a row of zeros, infinities and NaN in activations and weight scales, and a weight row of zeros among them."""
    import synth
    import torch_ggml_ops as tgo  # noqa: F401
    from torch_ggml_ops import _native

    qtype, lib = QTYPES[qname], _native.lib
    assert _native.forward_operand_for(qtype, rows, n) == "scaled"
    assert lib.tgo_forward_scratch_bytes_as(rows, k, n, qtype, _native.OPERANDS["scaled"]) > 0
    packed = synth.random_packed_weight(qtype, (n,), k, seed=qtype + n)
    packed[1] = 0
    # fp16 scale fields of a row's last block: an infinity, a NaN, and both in one row
    width, fields = synth.BLOCK_BYTES[qtype], synth._SCALE_FIELDS[qtype]
    for row, (first, last) in ((2, (0x7C00, 0x7C00)), (4, (0x7E00, 0x7E00)), (n - 1, (0xFC00, 0x7E01))):
        blocks = packed[row].view(-1, width)
        for block, value in ((0, first), (-1, last)):
            for field in fields:
                blocks[block, field], blocks[block, field + 1] = value & 0xFF, value >> 8
        if row == 4:
            blocks[0] = 0
    packed = packed.cuda()
    x = random_bf16((rows, k), seed=rows)
    x[3] = 0
    x[5, 256:] *= 2.0**-20
    x[6, :32] *= 2.0**-30
    x[8, 1] = float("nan")
    x[9] = float("nan")
    x[10, k - 1] = -float("inf")
    x[10, 0] = float("nan")
    x[rows - 1, 7] = float("inf")
    workspace = torch.empty(lib.tgo_q8_workspace_bytes(rows, k), dtype=torch.uint8, device="cuda")
    outputs = []
    for scratch_bytes in (0, lib.tgo_forward_scratch_bytes(rows, k, n, qtype)):
        scratch = torch.empty(max(scratch_bytes, 16), dtype=torch.uint8, device="cuda")
        # (whatever an earlier call left there must not be read)
        scratch.fill_(0xFF)
        workspace.fill_(0xFF)
        output = torch.empty((rows, n), dtype=torch.bfloat16, device="cuda")
        _native.check(
            lib.tgo_mmq_forward_scratch(
                x.data_ptr(), packed.data_ptr(), output.data_ptr(), workspace.data_ptr(), scratch.data_ptr() if scratch_bytes else None,
                rows, k, n, qtype, _native.stream_of(x.device),
            )
        )
        outputs.append(output)
    scaled, unpacked = outputs
    is_nan = scaled.isnan()
    assert torch.equal(is_nan, unpacked.isnan()) and not is_nan[rows // 2, n // 2]
    # (which of several NaN of a sum comes out is the instructions' business)
    assert torch.equal(scaled.view(torch.int16).masked_fill(is_nan, 0), unpacked.view(torch.int16).masked_fill(is_nan, 0))


@pytest.mark.parametrize("qname", ("Q5_K", "IQ2_S"))
@pytest.mark.parametrize("widths", [(2048, 512, 512), (2010, 500, 490, 70)])
def test_forward_of_several_projections(qname, widths):
    """One product over all columns: the bits of ``mmq_prepared``."""
    import synth
    import torch_ggml_ops as tgo
    from torch_ggml_ops import _native, prepared

    rows, k, qtype = 2000, 2048, QTYPES[qname]
    count = len(widths)
    assert prepared.multi_operand([qtype] * count, rows, widths) == "scaled"
    assert _native.lib.tgo_multi_forward_scratch_bytes(count, (ctypes.c_int64 * count)(*widths), (ctypes.c_int * count)(*[qtype] * count), rows, k) > 0
    packed = [synth.random_packed_weight(qtype, (n,), k, seed=3 + i).cuda() for i, n in enumerate(widths)]
    x = random_bf16((rows, k), seed=2)
    workspace = tgo.quantize_q8_1(x, "scaled")
    for output, weight, n in zip(tgo.mmq_multi(x, packed, [qtype] * count, widths), packed, widths):
        assert torch.equal(output, tgo.mmq_prepared(workspace, weight, rows, k, qtype, n, "scaled"))


def test_a_workspace_that_such_a_call_used_is_refused():
    """It holds the activations as the product reads them, whatever it held before: NaN where it is multiplied as a workspace, zeros where it is unpacked."""
    import synth
    import torch_ggml_ops as tgo
    from torch_ggml_ops import _native

    rows, n, k, qtype, lib = 2000, 2048, 2048, QTYPES["Q4_K"], _native.lib
    packed = synth.random_packed_weight(qtype, (n,), k, seed=1).cuda()
    x = random_bf16((rows, k), seed=1)
    workspace = tgo.quantize_q8_1(x, "scaled")
    assert torch.isfinite(tgo.mmq_prepared(workspace, packed, rows, k, qtype, n, "scaled").float()).all()
    scratch = torch.empty(lib.tgo_forward_scratch_bytes(rows, k, n, qtype), dtype=torch.uint8, device="cuda")
    output = torch.empty((rows, n), dtype=torch.bfloat16, device="cuda")
    stream = _native.stream_of(x.device)
    _native.check(lib.tgo_mmq_forward_scratch(x.data_ptr(), packed.data_ptr(), output.data_ptr(), workspace.data_ptr(), scratch.data_ptr(), rows, k, n, qtype,
                                              stream))
    assert torch.isfinite(output.float()).all()
    for kind in ("scaled", "int8"):
        assert torch.isnan(tgo.mmq_prepared(workspace, packed, rows, k, qtype, n, kind).float()).all()
    q = torch.ones(rows, k, dtype=torch.int8, device="cuda")
    d = torch.ones(rows, k // 32, device="cuda")
    s = torch.ones(rows, k // 32, device="cuda")
    _native.check(lib.tgo_q8_workspace_unpack(workspace.data_ptr(), q.data_ptr(), d.data_ptr(), s.data_ptr(), rows, k, stream))
    assert not q.any() and not d.any() and not s.any()
