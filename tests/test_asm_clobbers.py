"""Inline assembly of the kernels declares what it writes.

Scalar arithmetic (s_add_u32 and its like) writes SCC; the compiler may hold a carry or a
comparison in SCC across a statement that does not say so, and has scheduled such statements
between the two halves of a 64-bit address addition.
"""
import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "k100lc-rt4_amd" / "csrc"
SOURCES = sorted(p for p in CSRC.iterdir() if p.suffix in (".hip", ".h"))
WRITES_SCC = re.compile(r"\bs_(add|sub|and|or|xor|andn2|orn2|nand|nor|xnor|not|lsh[lr]|lshl\d_add|ashr|cmp|bitcmp|"
                        r"min|max|abs|absdiff|bfe|bcnt\w*|wqm|quadmask)\w*")


def asm_statements(text):
    for m in re.finditer(r"\basm\b\s*(?:volatile)?\s*\(", text):
        depth, i = 1, m.end()
        while depth:
            if text[i] == '"':
                i = re.compile(r'"(?:[^"\\]|\\.)*"').match(text, i).end()
                continue
            depth += {"(": 1, ")": -1}.get(text[i], 0)
            i += 1
        yield text[m.end():i - 1]


@pytest.mark.parametrize("path", SOURCES, ids=lambda p: p.name)
def test_asm_that_writes_scc_declares_it(path):
    for s in asm_statements(path.read_text()):
        if WRITES_SCC.search(s):
            assert '"scc"' in s, s


def test_dma_statements_are_seen():
    text = (CSRC / "rt4_dev.h").read_text()
    assert sum("s_add_u32 m0" in s and bool(WRITES_SCC.search(s)) for s in asm_statements(text)) == 2
