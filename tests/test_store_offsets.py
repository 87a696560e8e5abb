"""16-byte buffer stores take their whole offset in a vector register.

With a scalar offset the compiler leaves no wait state between a store of more than 8 bytes and a vector instruction that
overwrites the store's data registers, and gfx950 then stores parts of the new value."""
import pathlib
import re

import pytest

CSRC = pathlib.Path(__file__).resolve().parent.parent / "pyramidconvblock_amd" / "csrc"
SOURCES = sorted(p for p in CSRC.rglob("*") if p.suffix in (".h", ".hip") and "raw_buffer_store_b" in p.read_text())


def _arguments(text, at):
    """Top-level arguments of the call whose opening parenthesis is text[at]."""
    depth, parts, start = 0, [], at + 1
    for i in range(at, len(text)):
        c = text[i]
        if c in "([{":
            depth += 1
        elif c in ")]}":
            depth -= 1
            if depth == 0:
                return parts + [text[start:i].strip()]
        elif c == "," and depth == 1:
            parts.append(text[start:i].strip())
            start = i + 1
    raise AssertionError("unbalanced call")


@pytest.mark.parametrize("path", SOURCES, ids=lambda p: p.name)
def test_wide_stores_have_no_scalar_offset(path):
    text = path.read_text()
    for m in re.finditer(r"raw_buffer_store_b(?:96|128)\b\s*(?=\()", text):
        args = _arguments(text, m.end())
        assert args[3] == "0", f"{path.name}:{text[:m.start()].count(chr(10)) + 1}: scalar offset {args[3]}"


def test_there_are_such_stores():
    assert SOURCES
