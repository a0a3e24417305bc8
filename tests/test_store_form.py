"""The 12- and 16-byte buffer stores of the built library: none has a register
in its scalar offset.  The compiler keeps the wait states between such a store
and the next write of its data registers only where there is none."""
import os
import re
import shutil
import subprocess

import pytest

from igm_amd import _lib as L

STORE = re.compile(r"buffer_store_(?:format_\w+|dwordx[34]) (?:v|a)\[\d+:\d+\], (?:\S+, )?s\[\d+:\d+\], (\S+)")
OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"


def offending(text):
    """[(kernel, instruction)] of a disassembly."""
    bad, kernel, seen = [], None, 0
    for line in text.splitlines():
        if line.endswith(">:"):
            kernel = line.split("<")[1][:-2]
        m = STORE.search(line)
        seen += m is not None
        if m and re.match(r"(s|m|ttmp|vcc)", m.group(1)):
            bad.append((kernel, line.split("//")[0].strip()))
    return bad, seen


def test_the_pattern():
    text = ("0000 <k>:\n buffer_store_dwordx4 v[46:49], v115, s[84:87], s43 offen\n"
            " buffer_store_dwordx4 v[2:5], v45, s[92:95], 0 offen offset:16\n buffer_store_dword v2, v45, s[92:95], s4 offen\n"
            " buffer_store_dwordx3 a[2:4], off, s[92:95], m0\n buffer_store_dwordx4 v[2:5], v4, s[0:3], 64 offen\n")
    bad, seen = offending(text)
    assert [b[1].split()[-2:] for b in bad] == [["s43", "offen"], ["s[92:95],", "m0"]] and seen == 4


def test_no_wide_store_with_a_scalar_offset(tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    lib = shutil.copy(L.LIB_PATH, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=tmp_path, check=True, capture_output=True)
    objs = sorted(f for f in os.listdir(tmp_path) if f.endswith("gfx950"))
    assert objs
    total = 0
    for f in objs:
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", tmp_path / f], check=True, capture_output=True, text=True).stdout
        bad, seen = offending(text)
        total += seen
        assert not bad, (f, len(bad), bad[:3])
    assert total > 100
