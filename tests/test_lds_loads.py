"""The build's proof that hand-issued loads keep the wait states in front of them, on small functions: what it has to refuse and
what it has to let pass.  (The kernels themselves are checked by every build.)"""

import importlib.util
import sys
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "torch-ggml-ops_amd" / "csrc"


@pytest.fixture(scope="module")
def checker():
    sys.path.insert(0, str(CSRC))
    try:
        spec = importlib.util.spec_from_file_location("check_lds_loads", CSRC / "check_lds_loads.py")
        module = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(module)
    finally:
        sys.path.remove(str(CSRC))
    return module


def by_hand(*lines):
    return "\n".join(("\t;;#ASMSTART", *("\t" + line for line in lines), "\t;;#ASMEND"))


SLAB = "global_load_lds_dwordx4 v1, s[2:3]"
SOUND = by_hand("s_mov_b32 m0, s9", "s_nop 0", SLAB)


def problems(checker, lds, *lines):
    text = "\n".join(("\t.type\tkernel,@function", "kernel:  ; @kernel", *lines, "\ts_endpgm", ".Lfunc_end0:"))
    ((_, body, labels),) = checker.functions(text)
    return checker.check(body, labels, lds)[1]


@pytest.mark.parametrize(
    "lines",
    (
        (SOUND, SOUND),
        (by_hand("s_mov_b32 m0, s9", "s_nop 0", SLAB, SLAB + " offset:1024"),),
        ("\ts_add_u32 s9, s8, 16", SOUND),   # scalar results are interlocked
        ("\tv_readfirstlane_b32 s2, v9", "\ts_nop 2", SOUND),   # 3 + 2 wait states
        ("\tv_readfirstlane_b32 s4, v9", SOUND),
        ("\tv_readfirstlane_b32 s2, v9", "\ts_branch .LBB0_1", SOUND, ".LBB0_1:", "\tv_add_u32_e32 v5, v6, v7", "\ts_nop 0", SOUND),
    ),
)
def test_sound_code_passes(checker, lines):
    assert problems(checker, True, *lines) == []


@pytest.mark.parametrize(
    "lines",
    (
        (by_hand("s_mov_b32 m0, s9", SLAB),),
        (by_hand("s_mov_b32 m0, s9"), by_hand("s_nop 0", "s_nop 0", SLAB), by_hand(SLAB)),   # the second takes another's m0
        (SOUND, "\ts_mov_b32 m0, s5"),   # the compiler's own use of it
        (SOUND, by_hand("global_load_dwordx4 v[4:7], v1, s[2:3]")),   # not to LDS
        ("\tv_readfirstlane_b32 s3, v9", "\ts_nop 1", SOUND),   # 2 + 2 wait states
        ("\tv_mad_u64_u32 v[4:5], s[2:3], v3, s92, v[6:7]", SOUND),   # its carry
        ("\tv_cmp_eq_u32_e64 s[2:3], v4, v5", "\ts_cbranch_scc1 .LBB0_1", "\ts_nop 4", ".LBB0_1:", SOUND),   # a path around the wait
    ),
)
def test_missing_wait_states_are_refused(checker, lines):
    assert problems(checker, True, *lines)


def test_loads_to_registers(checker):
    load = by_hand("global_load_dwordx4 v[4:7], v1, s[2:3]")
    assert problems(checker, False, "\ts_mov_b32 m0, s5", load) == []
    assert problems(checker, False, "\tv_readlane_b32 s3, v9, 1", load)


def test_a_kernel_without_such_loads_is_refused(checker, tmp_path, monkeypatch):
    (tmp_path / "k.s").write_text("\t.type\tkernel,@function\nkernel:\n\ts_endpgm\n.Lfunc_end0:\n")
    for arguments in (("kernel", "1"), ("other", "1")):
        monkeypatch.setattr("sys.argv", ["check", str(tmp_path / "k.s"), "--kernel", arguments[0], "--expect", arguments[1]])
        assert checker.main() == 1
