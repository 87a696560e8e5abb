"""LDS reads that kernels wait for by hand (csrc/dense_wide.hip): no instruction touches a register that such a read is still on its way to.

The compiler takes a read in inline assembly to be done where it stands, and gives the register away once nothing uses the value any
more; the hardware does not order a read's return behind other writes of its register."""
import os
import pathlib
import re
import subprocess
import tempfile

import pytest

from test_store_offsets import OBJDUMP, _code_objects

INSTRUCTION = re.compile(r"\s+(\w+)(?:\s+(.*?))?\s*//\s*([0-9A-F]+):")
REGISTER = re.compile(r"\b([va])(?:(\d+)\b|\[(\d+):(\d+)\])")
KERNEL = re.compile(r"^[0-9a-f]* ?<(\w+)>:$", re.M)


def _registers(text):
    found = set()
    for bank, one, first, last in REGISTER.findall(text):
        found.update((bank, r) for r in (range(int(first), int(last) + 1) if first else (int(one),)))
    return found


def _parse(listing):
    """[(address, mnemonic, operands)] of a kernel's listing."""
    return [(int(m[3], 16), m[1], m[2] or "") for m in map(INSTRUCTION.match, listing.splitlines()) if m]


def _touched_in_flight(code):
    """Instructions that touch a register which an LDS read issued before them may still write.

    LDS operations end in order, so behind a wait for all but N of them those with N or more issued since are done; per register and program
    point the least number issued since its read, over all ways there."""
    index = {address: i for i, (address, _, _) in enumerate(code)}
    state, found, work = {0: {}}, {}, [0]
    while work:
        i = work.pop()
        flight = dict(state[i])
        while True:
            address, name, operands = code[i]
            is_lds = name.startswith("ds_")
            read = is_lds and not re.match(r"ds_(write|store|nop|(add|min|max|and|or|inc|dec)_[a-z0-9]+$)", name)
            target = _registers(operands.split(",")[0]) if read else set()
            # (a register that a later LDS read writes again is written in order)
            late = (_registers(operands.split(",", 1)[1]) if read and "," in operands else _registers(operands) - target) & flight.keys()
            if late:
                found[i] = (f"{address:x}", name, operands, sorted(late))
            if is_lds:
                flight = {r: n + 1 for r, n in flight.items() if n < 15}   # (no more than 15 can be outstanding)
                flight.update(dict.fromkeys(target, 0))
            elif name == "s_waitcnt":
                m = re.search(r"lgkmcnt\((\d+)\)", operands)
                if m:
                    flight = {r: n for r, n in flight.items() if n < int(m[1])}
            follow = []
            if name.startswith(("s_branch", "s_cbranch")):
                offset = int(operands.split()[0])
                follow.append(index[address + 4 + 4 * (offset - 0x10000 if offset >= 0x8000 else offset)])
            if name not in ("s_branch", "s_endpgm", "s_setpc_b64") and i + 1 < len(code):
                follow.append(i + 1)
            again = None
            for j in follow:
                known = state.get(j)
                if known is None:
                    state[j] = dict(flight)
                else:
                    less = {r: n for r, n in flight.items() if n < known.get(r, 99)}
                    if not less:
                        continue
                    known.update(less)
                if again is None:
                    again = j
                else:
                    work.append(j)
            if again is None:
                break
            i, flight = again, dict(state[again])
    return [found[i] for i in sorted(found)]


def _listing(lines):
    return _parse("\n".join(f"\t{text} // {address:012X}: 00000000" for address, text in lines))


def test_the_check_sees_a_register_given_away():
    read, wait = (0, "ds_read_b64_tr_b16 v[2:3], v9"), (12, "s_waitcnt lgkmcnt(0)")
    assert not _touched_in_flight(_listing([read, wait, (16, "v_mov_b32_e32 v2, v1"), (20, "s_endpgm")]))
    assert len(_touched_in_flight(_listing([read, (8, "v_mov_b32_e32 v2, v1"), wait, (20, "s_endpgm")]))) == 1
    # one read behind it may be outstanding, it may not; around a loop, that of the turn before
    behind = (8, "ds_read_b128 v[4:7], v9 offset:16")
    assert not _touched_in_flight(_listing([read, behind, (16, "s_waitcnt lgkmcnt(1)"), (20, "v_mov_b32_e32 v8, v3"), (24, "s_endpgm")]))
    assert len(_touched_in_flight(_listing([read, behind, (16, "s_waitcnt lgkmcnt(1)"), (20, "v_mov_b32_e32 v8, v4"), (24, "s_endpgm")]))) == 1
    loop = [(0, "v_mov_b32_e32 v8, v3"), (4, "ds_read_b64_tr_b16 v[2:3], v9"), (12, "s_cbranch_scc1 65532"), (16, "s_endpgm")]
    assert len(_touched_in_flight(_listing(loop))) == 1


def test_no_register_is_touched_while_a_read_is_on_its_way_to_it():
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump here")
    from pyramidconvblock_amd import _lib

    _lib.lib()   # (built if it has never been)
    checked, bad = 0, []
    for code in _code_objects(pathlib.Path(_lib.LIB_PATH)):
        if b"wide_gemm_k" not in code:
            continue
        with tempfile.NamedTemporaryFile(suffix=".co") as f:
            f.write(code)
            f.flush()
            text = subprocess.run([OBJDUMP, "-d", f.name], check=True, capture_output=True, text=True).stdout
        parts = KERNEL.split(text)
        for name, listing in zip(parts[1::2], parts[2::2]):
            instructions = _parse(listing)
            if any(n.startswith("ds_read") for _, n, _ in instructions):
                checked += 1
                bad += [(name, *hit) for hit in _touched_in_flight(instructions)]
    assert checked > 40 and not bad, (checked, len({b[0] for b in bad}), bad[:5])
