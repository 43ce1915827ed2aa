"""Inline assembly in the kernel sources tells the compiler every register it
writes: a register that is missing from the clobbers may hold a live value."""
import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "sheep_amd" / "csrc"


def statements(text):
    """The asm statements of a source, each as (instructions, operand lists)."""
    for m in re.finditer(r"\basm\b(?:\s+volatile)?\s*\(", text):
        depth, i, quoted = 1, m.end(), False
        while depth:
            c = text[i]
            if quoted:
                quoted, i = c != '"', i + (c == "\\")
            elif c == '"':
                quoted = True
            else:
                depth += (c == "(") - (c == ")")
            i += 1
        body = text[m.end():i - 1]
        code = re.match(r'(?:\s*"(?:[^"\\]|\\.)*")+', body).group()
        yield code, body[len(code):]


@pytest.mark.parametrize("src", sorted(p.name for p in CSRC.iterdir() if p.suffix in (".hip", ".h")))
def test_asm_that_writes_m0_says_so(src):
    for code, operands in statements((CSRC / src).read_text()):
        if re.search(r"\bs_\w+\s+m0\b", code):
            assert '"m0"' in operands.rsplit(":", 1)[-1], code
