"""Proves, on the assembly of one build, that hand-issued memory instructions keep the wait states that the hardware does not enforce.

    python3 check_lds_loads.py tgo_unpacked.s --kernel REGEX --expect 4 [--lds]

The compiler places the wait states between its own instructions, but does not look inside a piece of inline assembly.  Between the instruction
that writes and the hand-issued load that reads there have to lie, on every path,

  1 instruction    m0 written by the scalar unit, then a load to LDS, which takes its LDS address from m0
  5 instructions   a scalar register written by a vector instruction (readfirstlane, a comparison, a carry), then a load that names it

``s_nop N`` counts as N + 1.  --lds: the kernels' loads go to LDS; each of them has to have m0 written in its own piece of assembly, and nothing
outside of those may name m0, which is one of the compiler's reserved registers and therefore not protected by a clobber list.
"""

from __future__ import annotations

import argparse
import re
import sys

from check_loads_in_flight import functions

_SCALAR = re.compile(r"\bs(?:(\d+)|\[(\d+):(\d+)\])(?![\w.])")
_LOAD = re.compile(r"^(global|buffer|scratch|flat)_")
_ENDS = ("s_branch", "s_endpgm")   # nothing falls through them
M0_STATES, SCALAR_STATES = 1, 5


def _scalars(operands: str) -> frozenset:
    named = set()
    for single, first, last in _SCALAR.findall(operands):
        low, high = (int(single), int(single)) if single else (int(first), int(last))
        named.update(range(low, high + 1))
    if re.search(r"\bvcc\b", operands):
        named.add("vcc")
    return frozenset(named)


def _written_by_vector(mnemonic: str, operands: str) -> frozenset:
    """Scalar registers that a vector instruction may write: those among its first two operands."""
    if not mnemonic.startswith("v_"):
        return frozenset()
    parts = re.split(r",\s*", operands)
    # (a carry is the second operand; a mere source there makes the check stricter, not weaker)
    return _scalars(", ".join(parts[: 2 if re.search(r"_co_|v_mad_[iu]64|v_div_scale", mnemonic) else 1]))


def check(body, labels, lds: bool) -> tuple[int, list[str]]:
    """(hand-issued loads, violations) of one function."""
    sources = {}   # instruction -> those that may run right before it
    for at, (_, mnemonic, operands, _) in enumerate(body):
        if mnemonic in ("s_setpc_b64", "s_swappc_b64", "s_call_b64"):
            raise ValueError(f"{mnemonic} leaves the function: its paths cannot be followed")
        if not mnemonic.startswith(_ENDS):
            sources.setdefault(at + 1, []).append(at)
        if mnemonic.startswith(("s_branch", "s_cbranch")):
            sources.setdefault(labels[operands], []).append(at)

    def before(at, states):
        """(instruction, wait states between it and `at`) of all that run less than `states` wait states before it."""
        todo, seen = [(source, 0) for source in sources.get(at, ())], {}
        while todo:
            here, distance = todo.pop()
            if distance >= states or seen.get(here, states) <= distance:
                continue
            seen[here] = distance
            _, mnemonic, operands, _ = body[here]
            distance += int(operands, 0) + 1 if mnemonic == "s_nop" else 1
            todo += [(source, distance) for source in sources.get(here, ())]
        return seen

    issued, problems = 0, []
    for at, (number, mnemonic, operands, by_hand) in enumerate(body):
        if lds and not by_hand and re.search(r"\bm0\b", operands):
            problems.append(f"line {number}: {mnemonic} {operands} names m0 outside of the hand-issued loads")
        if not by_hand or not _LOAD.match(mnemonic):
            continue
        issued += 1
        if "_lds_" in mnemonic or operands.rstrip().endswith("lds"):
            for source in before(at, M0_STATES):
                if re.match(r"m0\b", body[source][2]):
                    problems.append(f"line {number}: {mnemonic} follows a write of m0 without a wait state")
            own = at   # its own piece of assembly writes m0
            while own >= 0 and body[own][3] == by_hand and not re.match(r"m0\b", body[own][2]):
                own -= 1
            if own < 0 or body[own][3] != by_hand:
                problems.append(f"line {number}: {mnemonic} takes m0 from elsewhere")
        elif lds:
            problems.append(f"line {number}: {mnemonic} does not go to LDS")
        named = _scalars(operands)
        for source in before(at, SCALAR_STATES):
            clash = _written_by_vector(body[source][1], body[source][2]) & named
            if clash:
                problems.append(f"line {number}: {mnemonic} {operands} too soon behind line {body[source][0]}: {body[source][1]} {body[source][2]}")
    return issued, problems


def main() -> int:
    parser = argparse.ArgumentParser()
    parser.add_argument("assembly")
    parser.add_argument("--kernel", required=True, help="regular expression that the mangled names of the kernels match")
    parser.add_argument("--expect", type=int, required=True, help="how many kernels must match")
    parser.add_argument("--lds", action="store_true", help="the hand-issued loads go to LDS")
    options = parser.parse_args()
    with open(options.assembly) as file:
        text = file.read()
    matched, failed = 0, False
    for name, body, labels in functions(text):
        if not re.search(options.kernel, name):
            continue
        matched += 1
        issued, problems = check(body, labels, options.lds)
        if issued == 0:
            problems.append("no hand-issued load found: the check cannot vouch for this kernel")
        for problem in problems:
            print(f"{options.assembly}: {name}: {problem}", file=sys.stderr)
        failed = failed or bool(problems)
    if matched != options.expect:
        print(f"{options.assembly}: {matched} kernels match {options.kernel}, expected {options.expect}", file=sys.stderr)
        failed = True
    return 1 if failed else 0


if __name__ == "__main__":
    sys.exit(main())
