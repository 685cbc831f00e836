"""Casts to the constant address space in device code (scalar loads of tables): the pointer must be one that
the kernel was given, never the address of a by-value argument or a local.  Those live in private memory as
the language has it, and only an optimised build happens to read them from the argument segment; the
unoptimised IR shows which of the two a cast is."""

import re
import shutil
import subprocess

import pytest

from holmes_amd import build as hb

SOURCES = sorted(p for p in hb.CSRC.glob("*.hip") if "address_space(4)" in p.read_text())


@pytest.mark.skipif(shutil.which(hb.HIPCC) is None, reason="hipcc is not installed")
@pytest.mark.parametrize("src", SOURCES, ids=lambda p: p.name)
def test_constant_address_casts_start_from_given_pointers(src, tmp_path):
    out = tmp_path / "device.ll"
    flags = [f for f in hb.FLAGS if not f.startswith("-O")]
    subprocess.run([hb.HIPCC, "-O0", *flags, "--cuda-device-only", "-S", "-emit-llvm", str(src), "-o", str(out)],
                   check=True, capture_output=True)
    defs, casts = {}, []
    for line in out.read_text().splitlines():
        if line.startswith("define"):
            defs = {}  # value names are per function
        m = re.match(r"\s*(%\S+) = (.*)", line)
        if not m:
            continue
        defs[m[1]] = m[2]
        c = re.match(r"addrspacecast ptr (\S+) to ptr addrspace\(4\)", m[2])
        if c:
            casts.append(defs.get(c[1], "an argument"))
    assert casts, "the source casts to the constant address space somewhere"
    assert all(d.startswith("load ptr") for d in casts), casts

