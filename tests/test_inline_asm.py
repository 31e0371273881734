"""Inline assembly of the kernels: what an instruction writes is declared to the compiler."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rzlinear_amd", "csrc")
# instructions that write their first operand and, where the name is in the second set, the scalar condition code
WRITES_FIRST = re.compile(r"\bs_(?:mov|add|sub|or|and|lshl|addc|cselect)\w*\s+(\w+)\s*,")
WRITES_SCC = re.compile(r"\bs_(?:add|sub|addc|and|or|lshl|cmp)\w*\s")


def statements():
    for name in sorted(os.listdir(CSRC)):
        if not name.endswith((".h", ".hip")):
            continue
        with open(os.path.join(CSRC, name)) as f:
            text = f.read()
        for m in re.finditer(r"asm volatile\((.*?)\);", text, re.S):
            yield "%s:%d" % (name, text.count("\n", 0, m.start()) + 1), m.group(1)


def test_the_loads_to_lds_are_found():
    assert sum("global_load_lds" in s for _, s in statements()) >= 3


@pytest.mark.parametrize("at,statement", list(statements()), ids=lambda v: v if "\n" not in v and len(v) < 40 else "")
def test_written_registers_are_clobbers_or_outputs(at, statement):
    template = re.match(r'\s*((?:"[^"]*"\s*)+)', statement).group(1)
    clobbers = statement.rsplit(":", 1)[-1]
    for register in WRITES_FIRST.findall(template):
        assert '"%s"' % register in clobbers, "%s writes %s" % (at, register)
    if WRITES_SCC.search(template):
        assert '"scc"' in clobbers, "%s writes scc" % at
