"""Proves, on the assembly of one build, that no register is touched while a hand-issued load is still writing it.

    python3 check_loads_in_flight.py tgo_backward.s --kernel REGEX --expect 5

The role-split grad-input kernel issues its prefetches in inline assembly and awaits them with counts of its own.  The compiler
takes the destination of such a load for valid at once: a copy, a spill or another use of the register before the wait would
be wrong without a word.  So every build follows all paths through those kernels and fails on the first
instruction that names a register whose hand-issued load may still be in flight.

The state that is followed is the list of outstanding loads, oldest first.  ``s_waitcnt vmcnt(N)`` completes all but the N
youngest (loads return in order).  Stores count in vmcnt as well; they are left out of the list, which can only make a load
look outstanding for longer.  Loads that the compiler issues itself take a place in the list and are otherwise its own business.
Every branch is taken both ways: code whose branches depend on one another has paths that no run can take, and the
kernel is written so that none of them leads around a load or its wait.
"""

from __future__ import annotations

import argparse
import re
import sys

_REGISTER = re.compile(r"\b([va])(?:(\d+)|\[(\d+):(\d+)\])(?![\w.])")
_LOAD = re.compile(r"^(global|buffer|scratch)_load")   # (flat loads return out of order: they are left out like stores)
_VMCNT = re.compile(r"vmcnt\((\d+)\)")
_QUEUE = 63   # vmcnt has six bits: the hardware holds a wave that would have more in flight


def _registers(operands: str) -> frozenset:
    named = set()
    for kind, single, first, last in _REGISTER.findall(operands):
        low, high = (int(single), int(single)) if single else (int(first), int(last))
        named.update((kind, i) for i in range(low, high + 1))
    return frozenset(named)


def functions(text: str):
    """(name, [(line number, mnemonic, operands, which piece of inline assembly, 0 for none)], {label: index}) of each function."""
    name, body, labels, by_hand, pieces = None, [], {}, 0, 0
    for number, line in enumerate(text.splitlines(), 1):
        stripped = line.strip()
        if stripped.startswith(";;#ASMSTART"):
            pieces += 1
            by_hand = pieces
        elif stripped.startswith(";;#ASMEND"):
            by_hand = 0
        code = stripped.split(";", 1)[0].strip()
        if not code:
            continue
        begins = re.match(r"\.type\s+(\S+),@function", code)
        if begins:
            name, body, labels = begins.group(1), [], {}
        elif name is None:
            continue
        elif code.startswith(".Lfunc_end"):
            yield name, body, labels
            name = None
        elif code.endswith(":"):
            labels[code[:-1]] = len(body)
        elif not code.startswith("."):
            mnemonic, _, operands = code.partition(" ")
            body.append((number, mnemonic, operands.strip(), by_hand))
    if name is not None:
        raise ValueError(f"{name} has no end")


def check(body, labels) -> tuple[int, list[str]]:
    """(hand-issued loads, violations) of one function."""
    issued = sum(by_hand != 0 and _LOAD.match(mnemonic) is not None for _, mnemonic, _, by_hand in body)
    problems, seen = {}, set()
    todo = [(0, ())]   # (instruction, outstanding loads: the registers of a hand-issued one, or None)
    while todo:
        at, queue = todo.pop()
        while True:
            while queue and queue[0] is None:   # (a load of the compiler's with nothing older to wait for)
                queue = queue[1:]
            if (at, queue) in seen:
                break
            seen.add((at, queue))
            if at >= len(body):
                raise ValueError("execution runs past the function's end")
            number, mnemonic, operands, by_hand = body[at]
            wait = _VMCNT.search(operands) if mnemonic == "s_waitcnt" else None
            if mnemonic == "s_waitcnt" and wait is None and "cnt(" not in operands:
                raise ValueError(f"line {number}: s_waitcnt in a form that is not read here: {operands}")
            if wait:
                left = int(wait.group(1))
                queue = queue[len(queue) - left :] if left < len(queue) else queue
            if by_hand and mnemonic.startswith("flat_"):
                raise ValueError(f"line {number}: a hand-issued {mnemonic} has no place in the order of the loads")
            touched = _registers(operands)
            if touched and any(entry is not None and entry & touched for entry in queue):
                problems.setdefault(number, f"line {number}: {mnemonic} {operands} names a register whose load is in flight")
                break
            if _LOAD.match(mnemonic) and not operands.rstrip().endswith("lds"):
                destination = _registers(operands.split(",", 1)[0]) if by_hand else None
                queue = (queue + (destination,))[-_QUEUE:]
            if mnemonic == "s_endpgm":
                break
            if mnemonic in ("s_setpc_b64", "s_swappc_b64", "s_call_b64", "s_cbranch_i_fork", "s_rfe_b64"):
                raise ValueError(f"line {number}: {mnemonic} leaves the function: its paths cannot be followed")
            if mnemonic == "s_branch":
                at = labels[operands]
                continue
            if mnemonic.startswith("s_cbranch"):
                todo.append((labels[operands], queue))
            at += 1
    return issued, [problems[number] for number in sorted(problems)]


def main() -> int:
    parser = argparse.ArgumentParser()
    parser.add_argument("assembly")
    parser.add_argument("--kernel", required=True, help="regular expression that the mangled names of the kernels match")
    parser.add_argument("--expect", type=int, required=True, help="how many kernels must match")
    options = parser.parse_args()
    with open(options.assembly) as file:
        text = file.read()
    matched, failed = 0, False
    for name, body, labels in functions(text):
        if not re.search(options.kernel, name):
            continue
        matched += 1
        issued, problems = check(body, labels)
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
