"""A load into LDS takes its destination from M0, and the ISA asks for one wait state between a scalar write of M0 and that load.
The compiler sees to it for its own instructions and cannot for those inside an asm statement, so each statement has to."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vla.cpp_amd", "csrc")


def asm_instructions(text):
    """The instructions of every asm statement of a source, as lists of texts."""
    for m in re.finditer(r'\basm\s*(?:volatile)?\s*\(\s*((?:"(?:[^"\\]|\\.)*"\s*)+)', text):
        string = "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', m.group(1)))
        yield [i.strip() for i in re.split(r"(?:\\n|\\t|;)+", string) if i.strip()]


def unsafe(instructions):
    """Loads into LDS with no wait state behind the M0 write in front of them, or no such write in their statement."""
    found, written = [], None  # instructions since M0 was written
    for i in instructions:
        if re.match(r"(global|buffer|scratch)_load_(lds_|.*\blds\b)", i):
            if written is None or written < 1:
                found.append(i)
        written = 0 if re.match(r"s_\w+ m0\b", i) else None if written is None else written + 1
    return found


def test_the_scan_knows_both_forms():
    bad = r'asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(b), "v"(p) : "memory");'
    good = r'asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(b));'
    assert [len(unsafe(i)) for t in (bad, good) for i in asm_instructions(t)] == [1, 0]


@pytest.mark.parametrize("path", sorted(glob.glob(os.path.join(CSRC, "*.h*"))), ids=os.path.basename)
def test_a_wait_state_stands_between_m0_and_the_load(path):
    with open(path) as f:
        for instructions in asm_instructions(f.read()):
            assert not unsafe(instructions), instructions


def test_loads_into_lds_are_among_them():
    with open(os.path.join(CSRC, "common.h")) as f:
        assert sum(any("_load_lds_" in i for i in s) for s in asm_instructions(f.read())) >= 4
