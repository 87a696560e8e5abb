"""16-byte buffer stores take their whole offset in a vector register.

With a scalar offset the compiler leaves no wait state between a store of more than 8 bytes and a vector instruction that
overwrites the store's data registers, and gfx950 then stores parts of the new value."""
import concurrent.futures
import os
import pathlib
import re
import struct
import subprocess
import tempfile

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


OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
WIDE_STORE = re.compile(r"buffer_store_dwordx[34]\s+v\[[\d:]+\], \S+ s\[[\d:]+\], (\w+)")   # data, offset, descriptor, scalar offset


def _code_objects(path):
    """The gfx950 code objects of a library: its offload bundles, one a source file."""
    data, magic = path.read_bytes(), b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        entries, = struct.unpack_from("<Q", data, at + len(magic))
        p = at + len(magic) + 8
        for _ in range(entries):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + length].decode()
            p += 24 + length
            if size and "gfx950" in name:
                yield data[at + offset:at + offset + size]
        at = data.find(magic, at + 1)


def _scalar_offsets(code):
    with tempfile.NamedTemporaryFile(suffix=".co") as f:
        f.write(code)
        f.flush()
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", f.name], check=True, capture_output=True, text=True).stdout
    return WIDE_STORE.findall(text)


def test_wide_stores_of_the_built_library_have_no_scalar_offset():
    """What the compiler made of it: every 12- and 16-byte buffer store of this library's own kernels."""
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump here")
    from pyramidconvblock_amd import _lib

    assert WIDE_STORE.findall("buffer_store_dwordx4 v[2:5], v6, s[8:11], s20 offen\nbuffer_store_dwordx3 v[2:4], off, s[8:11], 0 offset:16") == ["s20", "0"]
    _lib.lib()   # (built if it has never been)
    with concurrent.futures.ThreadPoolExecutor(4) as pool:
        offsets = [o for found in pool.map(_scalar_offsets, _code_objects(pathlib.Path(_lib.LIB_PATH))) for o in found]
    assert len(offsets) > 100 and set(offsets) == {"0"}, set(offsets)
