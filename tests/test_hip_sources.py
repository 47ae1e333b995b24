"""Inline assembly of the HIP sources names what it changes."""
from __future__ import annotations

import re
from pathlib import Path

HIP = Path(__file__).resolve().parents[1] / "unlimitedocr.c_amd" / "csrc" / "hip"


def asm_statements():
    for f in sorted(HIP.iterdir()):
        for m in re.finditer(r"\basm\s+(?:volatile\s*)?\((.*?)\)\s*;", f.read_text(), re.S):
            yield f.name, m.group(1)


def test_written_m0_is_a_clobber():
    """The compiler keeps values of its own in m0 (indexed registers, messages):
    a statement that sets m0 lists it."""
    seen = 0
    for name, text in asm_statements():
        code = "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', text.split("\n                 :")[0]))
        if re.search(r"\b[sv]_\w+ m0\b", code):
            seen += 1
            assert '"m0"' in text.rsplit(":", 1)[1], (name, text)
    assert seen > 0
