"""The build's proof that no register is touched while a hand-issued load is still writing it, on small functions: what it has
to refuse and what it has to let pass.  (The kernels themselves are checked by every build.)"""

import importlib.util
from pathlib import Path

import pytest

CHECKER = Path(__file__).resolve().parents[1] / "torch-ggml-ops_amd" / "csrc" / "check_loads_in_flight.py"


@pytest.fixture(scope="module")
def checker():
    spec = importlib.util.spec_from_file_location("check_loads_in_flight", CHECKER)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


def load(first, base="s[2:3]"):
    return f"\t;;#ASMSTART\n\tglobal_load_dwordx4 v[{first}:{first + 3}], v1, {base} offset:0x10\n\t;;#ASMEND"


def wait(count):
    return f"\t;;#ASMSTART\n\ts_waitcnt vmcnt({count})\n\t;;#ASMEND"


def problems(checker, *lines):
    text = "\n".join(("\t.type\tkernel,@function", "kernel:  ; @kernel", *lines, "\ts_endpgm", ".Lfunc_end0:"))
    ((name, body, labels),) = checker.functions(text)
    assert name == "kernel"
    return checker.check(body, labels)[1]


READ = "\tds_write_b128 v0, v[4:7]"
LOOP = (load(4), load(8), ".LBB0_1:", wait(1), READ, load(4), wait(1), "\tds_write_b128 v0, v[8:11]", load(8),
        "\ts_cbranch_scc1 .LBB0_1")


@pytest.mark.parametrize(
    "lines",
    (
        (load(4), wait(0), READ),
        (load(4), load(8), wait(1), READ),
        (load(4), "\tv_add_u32_e32 v20, v21, v22", "\ts_waitcnt vmcnt(0) lgkmcnt(0)", READ),   # one of the compiler's waits
        ("\tglobal_load_dword v4, v1, s[2:3]", "\tv_mov_b32_e32 v9, v4"),   # a load of the compiler's is its own business
        (load(4), "\tglobal_load_dword v30, v1, s[2:3]", wait(1), READ),   # and takes a place in the order
        LOOP,
    ),
)
def test_sound_code_passes(checker, lines):
    assert problems(checker, *lines) == []


@pytest.mark.parametrize(
    "lines",
    (
        (load(4), READ),
        (load(4), "\tv_mov_b32_e32 v40, v5", wait(0)),   # a copy of a live range that was split
        (load(4), "\tv_accvgpr_write_b32 a3, v7", wait(0)),
        (load(4), "\tscratch_store_dwordx4 off, v[4:7], off offset:16", wait(0)),   # a spill
        (load(4), "\tv_add_u32_e32 v6, v21, v22"),   # the register of a load that nobody reads, taken for something else
        (load(4), load(6)),
        (load(4), load(8), wait(2), READ),   # one load too few awaited
        (load(4), "\tglobal_store_dword v1, v2, s[2:3]", wait(1), READ),   # a store does not count for a younger load
        (load(4), "\tflat_load_dword v30, v[2:3]", wait(1), READ),
        (load(4), "\ts_cbranch_scc0 .LBB0_2", wait(0), ".LBB0_2:", READ),   # a path around the wait
        (*LOOP[:6], "\ts_cbranch_scc0 .LBB0_2", *LOOP[6:9], ".LBB0_2:", LOOP[9]),   # a path around a load: the next count is short
    ),
)
def test_register_in_flight_is_refused(checker, lines):
    assert problems(checker, *lines)


def test_what_cannot_be_followed_is_refused(checker, tmp_path, monkeypatch):
    for lines in (("\ts_setpc_b64 s[2:3]",), (load(4), "\ts_waitcnt 0x3f70", READ)):
        with pytest.raises(ValueError):
            problems(checker, *lines)
    # a kernel that matches but holds no such load, and a name that matches nothing
    text = "\t.type\tkernel,@function\nkernel:\n\ts_endpgm\n.Lfunc_end0:\n"
    (tmp_path / "k.s").write_text(text)
    for arguments in (("kernel", "1"), ("other", "1")):
        monkeypatch.setattr("sys.argv", ["check", str(tmp_path / "k.s"), "--kernel", arguments[0], "--expect", arguments[1]])
        assert checker.main() == 1
