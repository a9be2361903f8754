"""Registers that a store still reads.  On gfx950 a store of more than 64 bits takes its data from the registers after it has been issued; what overwrites them in the
next two wait states can be stored in its place.  The compiler keeps that distance, except behind a buffer store with a scalar register as its offset, where the
rows of Needleman-Wunsch's results came out mixed: so no kernel may store that way."""
import re
import struct
import subprocess
from pathlib import Path

import pytest

OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")


def _code_objects(library):
    """The gfx950 code objects in the bundles of a library's .hip_fatbin."""
    data, bundle = library.read_bytes(), b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(bundle)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + 24)
        entry = at + 32
        for _ in range(count if count < 16 else 0):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            if size and b"gfx950" in data[entry + 24:entry + 24 + length]:
                yield data[at + offset:at + offset + size]
            entry += 24 + length
        at = data.find(bundle, at + 24)


def _registers(operand):
    m = re.fullmatch(r"v\[(\d+):(\d+)\]|v(\d+)", operand)
    return set(range(int(m[1] or m[3]), int(m[2] or m[3]) + 1)) if m else set()


def _overwritten(lines):
    """(function, store, instruction) where a vector instruction writes a store's data less than two wait states after it."""
    function, stores = "", []
    for line in lines:
        if m := re.match(r"[0-9a-f]+ <(.*)>:", line):
            function, stores = m[1], []
            continue
        op, _, rest = line.split("//")[0].strip().partition(" ")
        operands = [o.strip() for o in rest.split(",")]
        if op.startswith("v_"):
            yield from ((function, text, line.strip()) for data, _, text in stores if data & _registers(operands[0]))
        if op in ("s_endpgm", "s_branch"):      # what follows in the listing does not follow in time
            stores = []
        states = int(operands[0], 0) + 1 if op == "s_nop" else 1
        stores = [(data, age + states, text) for data, age, text in stores if age + states < 2]
        if re.match(r"(buffer|global|flat|scratch)_store_dwordx[34]", op):
            stores.append((_registers(operands[0 if op.startswith("buffer") else 1]), 0, line.strip()))


def test_the_scan_sees_what_it_looks_for():
    store = "\tbuffer_store_dwordx4 v[4:7], v1, s[0:3], s8 offen // 0000: 00"
    found = lambda *lines: len(list(_overwritten(["0000 <kernel>:", *lines])))      # noqa: E731
    assert found(store, "\tv_add_u32_e32 v4, v2, v3") == found(store, "\ts_add_i32 s8, s8, 4", "\tv_pk_add_f16 v[6:7], v[0:1], v[2:3]") == 1
    assert found(store, "\tv_add_u32_e32 v8, v4, v5") == found(store, "\ts_nop 1", "\tv_mov_b32_e32 v4, 0") == found(store, "\ts_endpgm", "\tv_mov_b32_e32 v4, 0") == 0
    assert found("\tglobal_store_dwordx4 v[4:5], v[0:3], off", "\tv_mov_b32_e32 v3, 0") == 1 and found("\tglobal_store_dwordx2 v[4:5], v[0:1], off", "\tv_mov_b32_e32 v0, 0") == 0


def test_no_kernel_overwrites_what_a_store_reads(tmp_path):
    from lego_amd.runtime import LIB_PATH
    if not OBJDUMP.exists():
        pytest.skip("no llvm-objdump")
    functions = 0
    for code in _code_objects(LIB_PATH):
        path = tmp_path / "code.o"
        path.write_bytes(code)
        text = subprocess.run([str(OBJDUMP), "-d", "--no-show-raw-insn", "--mcpu=gfx950", str(path)], capture_output=True, text=True, check=True).stdout
        functions += text.count(">:\n")
        assert not list(_overwritten(text.split("\n")))
    assert functions > 100
