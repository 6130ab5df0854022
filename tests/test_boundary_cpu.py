"""CPU-only checks of the drop-in boundary: the C-ABI library loads and exports every symbol
declared in include/tgo.h, its argument checks fire before any launch, the Python
validators reproduce the reference's error contract (message fragments of
tests/test_mmq.py:176-223 and tests/test_grouped_mmq.py:483-561 in the reference), and the
operators' fake kernels / schemas are registered.  No kernel is launched here.
"""

import ctypes
import re
from pathlib import Path

import pytest
import torch

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def package():
    import torch_ggml_ops
    import synth
    from torch_ggml_ops import _native, _validate

    return torch_ggml_ops, _native, _validate, synth


def test_library_exports_every_declared_symbol(package):
    _, native, _, _ = package
    header = (ROOT / "include" / "tgo.h").read_text()
    declared = set(re.findall(r"\b(tgo_[a-z0-9_]+)\s*\(", header))
    assert declared, "no declarations found in include/tgo.h"
    for name in sorted(declared):
        assert hasattr(native.lib, name), f"{name} is declared but not exported"
    assert declared == set(native.EXPORTS)


def test_sizes_and_block_bytes(package):
    _, native, _, synth = package
    lib = native.lib
    assert lib.tgo_version() >= 110   # (the workspace grew with the scaled operands: callers size it through the library)
    for qtype, size in synth.BLOCK_BYTES.items():
        assert lib.tgo_block_bytes(qtype) == size
    assert lib.tgo_block_bytes(10) == 0
    # two bytes per value (fp16 operands) + two fp32 per 32 values + a power of two and 16 bytes of block sums per 256
    # values + a power of two per row, rows padded to 32, plus the 1 KiB tail
    assert lib.tgo_q8_workspace_bytes(33, 512) == 2 * 64 * 512 + 2 * 64 * 16 * 4 + 64 * 2 * (4 + 16) + 64 * 4 + 1024
    assert lib.tgo_q8_workspace_bytes(0, 512) == 0
    # the kind a call would use: scaled once it has 128 tiles of 256 rows x 128 outputs (both projections count)
    assert native.forward_operand() == "auto"
    assert native.forward_operand_for(13, 4096, 1024, 1) == "scaled"
    assert native.forward_operand_for(13, 4096, 1024 - 128, 1) == "int8"
    assert native.forward_operand_for(22, 512, 4096, 1) == "half"
    assert native.forward_operand_for(22, 2048, 1024, 2) == "scaled"
    assert lib.tgo_task_workspace_bytes(100, 7) % 16 == 0
    assert lib.tgo_task_workspace_bytes(100, 7) >= 4 * (1 + 3 * (13 + 7))


def test_the_kernels_of_a_call_are_named(package):
    """tgo_forward_kernel_for follows format, size, groups and setting, where tgo_forward_kernel_family sees rows and groups only."""
    _, native, _, _ = package
    assert native.forward_kernel_for(14, 64, 4096, 4096) == "tiles"
    assert native.forward_kernel_for(14, 64, 4096, 4099) == "mfma"         # no whole tiles of 16 weight rows
    assert native.forward_kernel_for(14, 64, 1024, 2048) == "mfma"         # fewer than four million weights
    assert native.forward_kernel_for(14, 129, 4096, 4096) == "mfma"
    assert native.forward_kernel_for(14, 1, 4096, 4096) == "gemv"
    assert native.forward_kernel_for(11, 1, 8192, 28672) == "tiles"
    assert native.forward_kernel_for(22, 8 * 64, 2048, 512, 64, 2) == "tiles"
    assert native.forward_kernel_for(22, 64 * 64, 2048, 512, 64, 2) == "mfma"
    assert native.forward_kernel_for(22, 8, 2048, 512, 256, 2) == "gemv"
    native.set_forward_operand("int8")
    try:
        assert native.forward_kernel_for(14, 64, 4096, 4096) == "mfma"     # the kind was asked for
        assert native.forward_kernel_for(22, 8 * 64, 2048, 512, 64, 2) == "mfma"
    finally:
        native.set_forward_operand("auto")
    for sizes in ((10, 1, 256, 16), (12, 0, 256, 16), (12, 1, 100, 16), (12, 1, 256, 0)):
        with pytest.raises(RuntimeError):
            native.forward_kernel_for(*sizes)


def test_rows_per_group_that_the_decode_kernel_takes(package):
    """By format, operand kind and, where skewed routing makes many tasks of one expert's weights, rows in all."""
    _, native, _, _ = package

    def most(qtype, groups, k, n, projections=1):
        rows = [r for r in range(5 * groups, 40 * groups, groups) if native.forward_kernel_for(qtype, r, k, n, groups, projections) == "tiles"]
        assert rows == list(range(5 * groups, 5 * groups + len(rows) * groups, groups))   # one line, nothing beyond it
        return rows[-1] // groups if rows else 4

    assert [most(q, 64, 2048, 512, 2) for q in (11, 12, 13, 14, 22)] == [16, 16, 16, 32, 12]
    assert [most(q, 256, 2048, 512, 2) for q in (11, 12, 13, 14, 22)] == [15, 10, 8, 15, 12]    # (15: scaled operands from 16 on)
    assert [most(q, 256, 512, 2048) for q in (11, 12, 13, 14, 22)] == [12, 10, 10, 7, 7]        # (scaled from 8 on)
    assert [most(q, 256, 1024, 4096) for q in (11, 12, 13, 14, 22)] == [6, 6, 6, 4, 4]          # (all scaled)
    assert [most(q, 128, 1024, 4096) for q in (11, 12, 13)] == [12, 10, 10]
    assert [most(q, 256, 4096, 1024, 2) for q in (11, 12, 13, 14, 22)] == [7, 7, 7, 7, 7]


def test_dense_rows_that_the_decode_kernel_takes(package):
    """By format, size and length of K: Q3_K, Q4_K, Q5_K, Q6_K, IQ2_S."""
    _, native, _, _ = package

    def most(n, k):
        found = []
        for qtype in (11, 12, 13, 14, 22):
            rows = [r for r in range(33, 200) if native.forward_kernel_for(qtype, r, k, n) == "tiles"]
            assert rows == list(range(33, 33 + len(rows)))   # one line, nothing beyond it
            found.append(rows[-1] if rows else 32)
        return found

    assert most(2048, 2048) == most(1024, 8192) == [128] * 5
    assert most(1024, 4096 - 256) == [32] * 5                      # fewer than four million weights
    assert most(4096, 4096) == [96, 96, 96, 64, 96]
    assert most(2048, 8192) == [96, 64, 64, 64, 96]
    assert most(1024, 16384) == [96, 32, 32, 64, 32]
    assert most(8192, 4096) == most(11008, 4096) == [64] * 5
    assert most(8192, 5120) == [64, 64, 48, 64, 64]
    assert most(14336, 4096) == [64, 48, 48, 64, 48]
    assert most(8192, 8192) == [64, 32, 32, 64, 48]
    assert most(4096, 14336) == [64, 32, 32, 64, 32]
    assert most(16384, 4096) == [64] * 5
    assert most(28672, 8192) == [32] * 5


def test_an_entry_point_reads_the_operand_setting_once():
    """The rules take the setting as an argument, and no function of the C ABI reads it twice: a change by another thread falls
    before or after a call, not into it."""
    csrc = ROOT / "torch-ggml-ops_amd" / "csrc"
    read = "forward_operand_setting()"
    for path in sorted(csrc.glob("*.h")):
        assert path.read_text().replace(f"int {read};", "").count(read) == 0, path.name
    functions = re.split(r"\n}\n|; }\n", (csrc / "tgo_api.hip").read_text())
    assert all(body.count(read) <= 1 for body in functions)
    others = [p for p in csrc.glob("*.hip") if p.name not in ("tgo_api.hip", "tgo_aux.hip")]
    assert all(read not in p.read_text() for p in others)


def test_c_abi_rejects_bad_arguments_before_launch(package):
    _, native, _, _ = package
    lib = native.lib
    fake = 0x10000  # never dereferenced: every call below fails its checks first
    assert lib.tgo_mmq_forward(fake, fake, fake, fake, 0, 256, 8, 12, None) == 1
    assert b"zero-row" in lib.tgo_last_error()
    assert lib.tgo_mmq_forward(fake, fake, fake, fake, 4, 300, 8, 12, None) == 1
    assert b"multiple of 256" in lib.tgo_last_error()
    assert lib.tgo_mmq_forward(fake, fake, fake, fake, 4, 256, 8, 10, None) == 1
    assert b"unsupported quant_type" in lib.tgo_last_error()
    assert lib.tgo_mmq_forward(fake, fake + 2, fake, fake, 4, 256, 8, 12, None) == 1
    assert b"16-byte aligned" in lib.tgo_last_error()
    assert lib.tgo_mmq_grad_input(None, fake, fake, fake, 4, 8, 256, 12, None) == 1
    assert b"must not be null" in lib.tgo_last_error()
    assert lib.tgo_grouped_mmq_forward(fake, fake, None, fake, None, fake, fake, fake, 4, 256, 8, 2, 3, 12, None) == 1
    assert b"active expert count exceeds" in lib.tgo_last_error()
    assert lib.tgo_grouped_mmq_forward(fake, fake, fake, fake, None, fake, fake, fake, 4, 256, 8, 4, 3, 12, None) == 1
    assert b"given together" in lib.tgo_last_error()
    total, count = ctypes.c_double(), ctypes.c_int64()
    assert lib.tgo_profile_read(99, ctypes.byref(total), ctypes.byref(count)) == 1


def test_dense_validation_messages(package):
    _, _, validate, synth = package
    validate.REQUIRE_DEVICE = False
    try:
        packed = synth.random_packed_weight(12, (37,), 2048, seed=1)
        x = torch.randn(4, 2048).to(torch.bfloat16)
        assert validate.dense(x, packed, 12, 37, backward=False) == (4, 2048, 37)
        assert validate.dense(torch.randn(2, 3, 37).to(torch.bfloat16), packed, 12, 2048, backward=True) == (6, 2048, 37)
        cases = [
            (lambda: validate.dense(x[:, ::2], packed, 12, 37, backward=False), "contiguous"),
            (lambda: validate.dense(x[1:], packed, 12, 37, backward=False), "zero storage offset"),
            (lambda: validate.dense(x, packed.reshape(-1)[:-1].clone(), 12, 37, backward=False), "expected"),
            (lambda: validate.dense(x, packed, 10, 37, backward=False), "unsupported quant_type"),
            (lambda: validate.dense(x[:0], packed, 12, 37, backward=False), "zero-row"),
            (lambda: validate.dense(x.float(), packed, 12, 37, backward=False), "torch.bfloat16"),
            (lambda: validate.dense(x, packed.to(torch.int8), 12, 37, backward=False), "torch.uint8"),
            (lambda: validate.dense(x[:, :300].contiguous(), packed, 12, 37, backward=False), "multiple of 256"),
            (lambda: validate.dense(x, packed, 12, 0, backward=False), "out_features must be positive"),
            (lambda: validate.dense(x[:, :37].contiguous(), packed, 12, 2000, backward=True), "multiple of 256"),
            (lambda: validate.dense(x[:0, :37].contiguous(), packed, 12, 2048, backward=True), "zero-row"),
        ]
        for call, fragment in cases:
            with pytest.raises(RuntimeError, match=fragment):
                call()
    finally:
        validate.REQUIRE_DEVICE = True
    with pytest.raises(RuntimeError, match="CUDA/HIP tensor"):
        validate.dense(x, packed, 12, 37, backward=False)


def test_grouped_validation_messages(package):
    _, _, validate, synth = package
    validate.REQUIRE_DEVICE = False
    try:
        packed = synth.random_packed_weight(12, (8, 37), 2048, seed=2)
        x = torch.randn(262, 2048).to(torch.bfloat16)
        experts = torch.tensor([0, 2, 5, 7], dtype=torch.int64)
        offsets = torch.tensor([1, 128, 257, 262], dtype=torch.int32)
        shape = validate.grouped(x, packed, experts, offsets, 12, 37, backward=False)
        assert shape == (262, 2048, 37, 8, 4, 37 * 8 * 144)
        cases = [
            (lambda: validate.grouped(x[:, ::2], packed, experts, offsets, 12, 37, backward=False), "contiguous"),
            (lambda: validate.grouped(x[1:], packed, experts, offsets, 12, 37, backward=False), "zero storage offset"),
            (lambda: validate.grouped(x, packed[:, :, :-1].contiguous(), experts, offsets, 12, 37, backward=False), "bytes per row"),
            (lambda: validate.grouped(x, packed, experts, offsets, 10, 37, backward=False), "unsupported quant_type"),
            (lambda: validate.grouped(x[:0], packed, experts, offsets, 12, 37, backward=False), "zero-row"),
            (lambda: validate.grouped(x, packed, experts, offsets.long(), 12, 37, backward=False), "torch.int32"),
            (lambda: validate.grouped(x, packed, experts.int(), offsets, 12, 37, backward=False), "torch.int64"),
            (lambda: validate.grouped(x, packed, experts[:3], offsets, 12, 37, backward=False), "equal lengths"),
            (lambda: validate.grouped(x, packed[0], experts, offsets, 12, 37, backward=False), r"\[experts, out_features, row_bytes\]"),
            (lambda: validate.grouped(x, packed, experts, offsets, 12, 38, backward=False), "does not match out_features"),
            (lambda: validate.grouped(x, packed[:3].contiguous(), experts, offsets, 12, 37, backward=False), "active expert count exceeds"),
            (lambda: validate.grouped(x[:, :37].contiguous(), packed, experts, offsets, 12, 2000, backward=True), "multiple of 256"),
        ]
        for call, fragment in cases:
            with pytest.raises(RuntimeError, match=fragment):
                call()
    finally:
        validate.REQUIRE_DEVICE = True


def test_second_weight_of_a_pair_is_checked_like_the_first(package):
    """A second weight with the first one's geometry needs no second pass through the checks; any other goes through
    them and fails with their message (or with the pair's own, when it is a valid weight of another expert count)."""
    from torch_ggml_ops.grouped_mmq import _forward

    _, _, validate, synth = package
    validate.REQUIRE_DEVICE = False
    try:
        packed = synth.random_packed_weight(12, (8, 37), 2048, seed=2)
        other = synth.random_packed_weight(12, (8, 37), 2048, seed=3)
        assert validate.same_weight_geometry(packed, other)
        assert not validate.same_weight_geometry(packed, other[:, :, :-1])                  # not contiguous
        assert not validate.same_weight_geometry(packed, other[:4].contiguous())           # fewer experts
        assert not validate.same_weight_geometry(packed, other.to(torch.int8))             # another dtype
        assert not validate.same_weight_geometry(packed, other.reshape(-1)[16:].reshape(-1))   # another shape, offset
        x = torch.randn(262, 2048).to(torch.bfloat16)
        experts = torch.tensor([0, 2, 5, 7], dtype=torch.int64)
        offsets = torch.tensor([1, 128, 257, 262], dtype=torch.int32)
        cases = [
            (other[:, :, :-1], "contiguous"),
            (other[:, :36].contiguous(), "does not match out_features"),
            (other.to(torch.int8), "torch.uint8"),
            (other[:4].contiguous(), "identical physical geometry"),
        ]
        for second, fragment in cases:
            with pytest.raises(RuntimeError, match=fragment):
                _forward(x, packed, second, experts, offsets, 12, 37)
    finally:
        validate.REQUIRE_DEVICE = True


def test_operator_schemas_and_fake_kernels(package):
    tgo, _, _, _ = package
    ops = torch.ops.torch_ggml_ops
    assert str(ops.mmq.default._schema) == (
        "torch_ggml_ops::mmq(Tensor input, Tensor packed_weight, int quant_type, int out_features) -> Tensor"
    )
    assert "-> (Tensor, Tensor)" in str(ops.grouped_mmq_pair.default._schema)
    x = torch.empty(3, 5, 512, dtype=torch.bfloat16, device="meta")
    w = torch.empty(37, 288, dtype=torch.uint8, device="meta")
    assert tgo.mmq(x, w, 12, 37).shape == (3, 5, 37)
    assert ops.mmq_grad_input.default(torch.empty(3, 5, 37, dtype=torch.bfloat16, device="meta"), w, 12, 512).shape == (3, 5, 512)
    rows = torch.empty(20, 512, dtype=torch.bfloat16, device="meta")
    experts = torch.empty(8, 37, 288, dtype=torch.uint8, device="meta")
    indices = torch.empty(4, dtype=torch.int64, device="meta")
    offsets = torch.empty(4, dtype=torch.int32, device="meta")
    assert tgo.grouped_mmq(rows, experts, indices, offsets, 12, 37).shape == (20, 37)
    first, second = tgo.grouped_mmq_pair(rows, experts, experts, indices, offsets, 12, 37)
    assert first.shape == second.shape == (20, 37)
    grad = torch.empty(20, 37, dtype=torch.bfloat16, device="meta")
    assert ops.grouped_mmq_grad_input.default(grad, experts, indices, offsets, 12, 512).shape == (20, 512)
    assert ops.grouped_mmq_pair_grad_input.default(grad, grad, experts, experts, indices, offsets, 12, 512).shape == (20, 512)


def test_cpu_tensors_have_no_fallback(package):
    tgo, _, _, synth = package
    packed = synth.random_packed_weight(12, (4,), 256, seed=3)
    x = torch.randn(2, 256).to(torch.bfloat16)
    with pytest.raises(NotImplementedError):
        tgo.mmq(x, packed, 12, 4)


def test_synthetic_generators_are_seeded_and_well_formed(package, oracle):
    _, _, _, synth = package
    import numpy as np

    for qtype in synth.BLOCK_BYTES:
        first = synth.random_packed_weight(qtype, (3, 5), 512, seed=11)
        again = synth.random_packed_weight(qtype, (3, 5), 512, seed=11)
        assert torch.equal(first, again) and first.shape == (3, 5, synth.row_bytes(qtype, 512))
        values = oracle.dequant_f32(qtype, first.numpy(), 512)
        assert np.isfinite(values).all()
    tokens, indices, offsets, weights = synth.zipf_routing(64, 16, 4, seed=5)
    assert tokens.numel() == 256 == int(offsets[-1]) and weights.numel() == 256
    assert (indices[1:] > indices[:-1]).all() and (offsets[1:] > offsets[:-1]).all()


def test_token_runs_drop_rows_outside_the_input(package):
    """The host half of the per-token sum behind the gathered operators' gradients: the rows listed token by token in
    row order, with the rows whose index lies outside the token range behind the last run (the kernel that adds the
    runs up never sees them).  Summing the runs on the CPU gives the per-token sums."""
    from torch_ggml_ops.gathered import _token_runs

    grad_rows = torch.arange(24, dtype=torch.float32).reshape(6, 4).to(torch.bfloat16)
    row_index = torch.tensor([2, -1, 0, 9, 3, 2])
    order, starts = _token_runs(row_index, 4)
    assert order.dtype == torch.int64 and starts.dtype == torch.int64
    assert starts.tolist() == [0, 1, 1, 3, 4]
    assert order.tolist()[:4] == [2, 0, 5, 4] and sorted(order.tolist()[4:]) == [1, 3]
    result = torch.zeros(4, 4)
    for token in range(4):
        for row in order[starts[token]:starts[token + 1]].tolist():
            result[token] += grad_rows[row].float()
    expected = torch.zeros(4, 4)
    for row, token in enumerate(row_index.tolist()):
        if 0 <= token < 4:
            expected[token] += grad_rows[row].float()
    torch.testing.assert_close(result, expected, rtol=0, atol=0)


def test_loss_of_no_rows_is_zero(package):
    """No row, no chunk: the mean over at least one row of nothing, and an empty gradient.  (No kernel is involved.)"""
    tgo, _, _, synth = package
    weight = synth.random_packed_weight(synth.Q4_K, (64,), 256, seed=1)
    hidden = torch.zeros(0, 256, dtype=torch.bfloat16, requires_grad=True)
    targets = torch.zeros(0, dtype=torch.int64)
    loss = tgo.chunked_lm_head_loss(hidden, weight, targets, synth.Q4_K, 64)
    assert loss.shape == () and loss.dtype == torch.float32 and loss.item() == 0.0
    (loss * 2).backward()
    assert hidden.grad.shape == (0, 256) and hidden.grad.dtype == torch.bfloat16
    assert not tgo.chunked_lm_head_loss(hidden.detach(), weight, targets, synth.Q4_K, 64).requires_grad


@pytest.mark.parametrize("case", ("here", "missing", "another torch"))
def test_package_loads_without_the_direct_calls(case, tmp_path):
    """_direct.so belongs to one torch and one Python: without it, or with another torch, the package says so and sends every
    call through the registered operators."""
    import shutil
    import subprocess
    import sys

    package = tmp_path / "torch_ggml_ops"
    shutil.copytree(ROOT / "torch-ggml-ops_amd" / "torch_ggml_ops", package)
    if case == "missing":
        (package / "_direct.so").unlink()
    program = (
        "import torch, warnings\n"
        + ("torch.__version__ = '9.9.0'\n" if case == "another torch" else "")
        + "with warnings.catch_warnings(record=True) as seen:\n"
        "    warnings.simplefilter('always')\n"
        "    import torch_ggml_ops as tgo\n"
        "from torch_ggml_ops import _native\n"
        f"assert tgo.__file__.startswith({str(tmp_path)!r})\n"
        "messages = [str(w.message) for w in seen if 'torch_ggml_ops' in str(w.message)]\n"
        f"assert (_native.direct is not None) == (not messages) == {case == 'here'}, (_native.direct, messages)\n"
        "x, w = torch.zeros(2, 256, dtype=torch.bfloat16), torch.zeros(3, 144, dtype=torch.uint8)\n"
        "try:\n"
        "    tgo.mmq(x, w, 12, 3)\n"
        "except NotImplementedError as error:\n"
        "    assert 'torch_ggml_ops::mmq' in str(error)\n"
        "else:\n"
        "    raise AssertionError('a call on the CPU went through')\n"
    )
    done = subprocess.run([sys.executable, "-c", program], cwd=tmp_path, capture_output=True, text=True, timeout=100)
    assert done.returncode == 0, done.stderr


def test_multi_forward_rejects_missing_arrays(package):
    _, native, _, _ = package
    lib, fake = native.lib, 0x10000
    one = dict(packed=(ctypes.c_void_p * 1)(fake), out=(ctypes.c_void_p * 1)(fake), n=(ctypes.c_int64 * 1)(8), q=(ctypes.c_int * 1)(12))
    for missing in one:
        given = {**one, missing: None}
        status = lib.tgo_mmq_multi_forward(
            fake, 1, given["packed"], given["out"], given["n"], given["q"], fake, None, 4, 256, 0, None
        )
        assert status == 1 and b"must not be null" in lib.tgo_last_error()


def test_scratch_of_split_calls_has_to_be_aligned(package):
    """The kernels store 16 bytes at a time into it.  (Calls that need none may be given any pointer.)"""
    _, native, _, _ = package
    lib, fake = native.lib, 0x10000
    rows, k, n, qtype = 64, 4096, 1024, 13
    assert lib.tgo_forward_scratch_bytes(rows, k, n, qtype) > 0
    out, sizes, types = (ctypes.c_void_p * 1)(fake), (ctypes.c_int64 * 1)(n), (ctypes.c_int * 1)(qtype)
    for status in (
        lib.tgo_mmq_forward_scratch(fake, fake, fake, fake, fake + 8, rows, k, n, qtype, None),
        lib.tgo_mmq_forward_prepared_scratch(fake, fake, fake, fake + 8, rows, k, n, qtype, 0, None),
        lib.tgo_mmq_multi_forward(fake, 1, out, out, sizes, types, fake, fake + 8, rows, k, 0, None),
    ):
        assert status == 1 and b"scratch data pointer must be 16-byte aligned" in lib.tgo_last_error()


def test_helper_operators_check_what_they_are_given(package, monkeypatch):
    """The registered operators behind the backward passes and the loss, called as a user may call them: a tensor of another
    type, shape, device or layout never reaches a kernel."""
    _, _, validate, synth = package
    from torch_ggml_ops import lm_head, moe, prepared

    monkeypatch.setattr(validate, "REQUIRE_DEVICE", False)
    rows, grad = torch.zeros(6, 16, dtype=torch.bfloat16), torch.zeros(3, 16, dtype=torch.bfloat16)
    slots, weights = torch.zeros(3, 2, dtype=torch.int64), torch.zeros(3, 2)
    hidden, targets = torch.zeros(4, 256, dtype=torch.bfloat16), torch.zeros(4, dtype=torch.int64)
    packed = synth.random_packed_weight(synth.Q4_K, (8,), 256, seed=1)
    elsewhere = torch.zeros(3, 2, dtype=torch.int64, device="meta")

    def refused(function, *arguments, match):
        with pytest.raises(RuntimeError, match=match):
            function(*arguments)

    for arguments, match in (
        ((rows.float(), grad, slots), "rows must have dtype torch.bfloat16"),
        ((rows, grad.float(), slots), "grad_tokens must have dtype torch.bfloat16"),
        ((rows, grad, slots.int()), "slot_rows must have dtype torch.int64"),
        ((rows, grad, elsewhere), "same device"),
        ((rows, grad[:2], slots), "grad_tokens must have shape"),
        ((rows, grad[:, :8].contiguous(), slots), "grad_tokens must have shape"),
        ((rows, grad, slots[:, 0].contiguous()), "slot_rows must have shape"),
        ((rows[0], grad, slots), "rows must have shape"),
        ((rows.t().contiguous().t(), grad, slots), "rows must be contiguous"),
        ((rows, grad.t().contiguous().t(), slots), "grad_tokens must be contiguous"),
        ((rows, grad, slots.t().contiguous().t()), "slot_rows must be contiguous"),
        ((rows[:, :12].contiguous(), grad[:, :12].contiguous(), slots), "multiple of 8"),
    ):
        refused(moe._check_weight_grad, *arguments, match=match)
    for arguments, match in (
        ((slots.int(), weights, 6), "slot_rows must have dtype torch.int64"),
        ((slots, weights.double(), 6), "slot_weights must have dtype torch.float32"),
        ((slots, weights[:2], 6), "must both have shape"),
        ((slots[0], weights[0], 6), "must both have shape"),
        ((slots, weights.t().contiguous().t(), 6), "slot_weights must be contiguous"),
        ((elsewhere, weights, 6), "same device"),
        ((slots, weights, 0), "num_rows must be positive"),
    ):
        refused(moe._check_inverse, *arguments, match=match)
    for bad, match in ((targets[:3], "one entry per row"), (targets.int(), "one entry per row"), (targets.reshape(2, 2), "one entry per row")):
        refused(lm_head._check_loss, hidden, bad, 256, match=match)
    refused(lm_head._check_loss, hidden, targets, 0, match="chunk_rows")
    one = torch.ones(())
    for arguments, match in (
        ((hidden.float(), one), "input must have dtype torch.bfloat16"),
        ((hidden, one.double()), "factor must have dtype torch.float32"),
        ((hidden, torch.ones(2)), "factor must have one element"),
        ((hidden.t().contiguous().t(), one), "input must be contiguous"),
        ((hidden, one.to("meta")), "same device"),
    ):
        refused(lm_head._check_scale, *arguments, match=match)
    for arguments in (([packed], [12, 12], [8]), ([packed], [12], [8, 8]), ([packed, packed], [12], [8]), ([], [], [])):
        with pytest.raises(ValueError, match="equal length"):
            prepared._check_projections(*arguments)


def test_version_is_the_headers(package):
    """And the header's has grown past 112, the last one without the entry points that the list below begins with."""
    _, native, _, _ = package
    header = (ROOT / "include" / "tgo.h").read_text()
    version = int(re.search(r"#define TGO_VERSION (\d+)", header).group(1))
    assert native.lib.tgo_version() == version >= 113
    for name in ("tgo_forward_scratch_bytes", "tgo_mmq_multi_forward", "tgo_mmq_pair_grad_input", "tgo_route", "tgo_lm_head_loss"):
        assert f"{name}(" in header


def test_gradient_workspace_without_a_cotangent_that_is_not_packed(package):
    """Calls that unpack their weights read cotangents of whole stages as they stand: room for the weights is all that they ask for."""
    _, native, _, _ = package
    lib = native.lib
    both = (ctypes.c_int64 * 2)(2048, 512)
    assert lib.tgo_dense_grad_workspace_bytes(16384, 28672, 1024, 12) == 2 * 28672 * 1024
    assert lib.tgo_multi_grad_workspace_bytes(2, both, 4096, 2048) == 2 * 2560 * 2048
    assert lib.tgo_pair_grad_workspace_bytes(4096, 2048, 2048, 14) == 2 * 2 * 2048 * 2048
    assert lib.tgo_dense_grad_workspace_bytes(4096, 2047, 2048, 12) == 2 * 2048 * 2048 + 2 * 4096 * 2048   # (both packed)


def test_gradients_that_unpack_their_weights_once(package):
    """Not where that measured slower: long reductions over a few columns, which wait for their cotangent, and pairs of one shape, which are one call
    otherwise too."""
    _, native, _, _ = package

    def unpacks(rows, widths, k):
        return native.lib.tgo_multi_grad_workspace_bytes(len(widths), (ctypes.c_int64 * len(widths))(*widths), rows, k) > 0

    for rows, widths, k in ((4096, [28672], 512), (3193, [15872], 768), (2048, [8192], 1536), (195, [832, 832], 2560), (2857, [5632, 5632], 1024)):
        assert not unpacks(rows, widths, k)
    for rows, widths, k in ((4096, [4096], 2048), (2048, [4096, 1024, 1024], 4096), (161, [2188, 547, 547], 1280), (8192, [15872], 512), (4096, [2048, 2048], 2048)):
        assert unpacks(rows, widths, k)


def test_forward_calls_that_unpack_their_weights_once(package):
    """Not short reductions of a few hundred rows, whose activations the other kernels quantize in less time than the rule once held against them."""
    _, native, _, _ = package

    def unpacks(qtype, rows, n, k):
        return native.lib.tgo_forward_scratch_bytes_as(rows, k, n, qtype, native.OPERANDS["scaled"]) > 0

    for call in ((11, 123, 18688, 512), (12, 320, 18752, 512), (11, 463, 9216, 768), (13, 374, 11281, 512)):
        assert not unpacks(*call)
    for call in ((12, 4096, 4096, 4096), (12, 2000, 2048, 2048), (13, 4096, 4096, 2048), (11, 2424, 13878, 3584)):
        assert unpacks(*call)
