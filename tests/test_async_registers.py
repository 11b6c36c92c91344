"""Loads and atomics whose result is a register are the compiler's to wait for.  An assembly statement that issues one and leaves the wait to a later
statement gives the compiler a register that it takes for written: it may copy or spill the old value in between, silently."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flash-moba_amd", "csrc")
FAMILIES = {  # an instruction that writes a register later, the counter that says when
    "atomic": (r"(global|flat|buffer)_atomic_\w+[^\\]* (sc0|glc)", "vmcnt"),
    "lds": (r"ds_(read|bpermute|permute|swizzle|\w+_rtn)", "lgkmcnt"),
    "load": (r"(global|flat|buffer|scratch)_load_(?!lds)", "vmcnt"),
}


def _asm_statements(text):
    for m in re.finditer(r"\basm\s*(volatile)?\s*\(", text):
        depth, i, quoted = 1, m.end(), False
        while depth:
            c = text[i]
            quoted ^= c == '"' and text[i - 1] != "\\"
            depth += 0 if quoted else (c == "(") - (c == ")")
            i += 1
        yield text.count("\n", 0, m.start()) + 1, text[m.end():i - 1]


def _unawaited(text, family):
    instr, counter = FAMILIES[family]
    for line, body in _asm_statements(text):
        last = None
        for last in re.finditer(instr, body):
            pass
        if last and not re.search(r"s_waitcnt[^\\]*%s\(0\)" % counter, body[last.end():]):
            yield line


@pytest.mark.parametrize("family", sorted(FAMILIES))
def test_no_statement_leaves_a_register_on_its_way(family):
    files = sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h")))
    assert files
    found = ["%s:%d" % (os.path.basename(f), n) for f in files for n in _unawaited(open(f).read(), family)]
    assert not found


def test_the_search_finds_one():
    stmt = 'asm volatile("%s" : "=v"(x) : "v"(p) : "memory");'
    assert list(_unawaited(stmt % "global_load_dword %0, %1, off", "load")) == [1]
    assert not list(_unawaited(stmt % "global_load_dword %0, %1, off\\n\\ts_waitcnt vmcnt(0)", "load"))
    assert not list(_unawaited(stmt % "global_load_lds_dwordx4 %0, off", "load"))
