"""Addresses of the row-parallel LD solves (k_tri_chain_rp, k_tri_chain_rpf),
read from the compiled kernels on the CPU.

Lanes past the last row of a piece read on, past the last row of all beyond
the buffer, and count on the hardware to return 0 there.  It compares the
vector offset of the access with the buffer's size; a scalar offset is not
part of that comparison (or is subtracted from the size first, which wraps
round where it is the larger one), so none of these accesses may have one."""
from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

import sc23ad as S

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
KERNEL = re.compile(r"^[0-9a-f]+ <(\S*k_tri_chain_rpf?I\S*)>:")
ANY = re.compile(r"^[0-9a-f]+ <(\S+)>:")
# buffer_load_dwordx4 v[2:5], v1, s[4:7], 0 offen offset:16
ACCESS = re.compile(r"^\s+(buffer_\S+) [^,]+, (?:v\d+|off), s\[\d+:\d+\], (\S+)")


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="llvm-objdump not found")
def test_buffer_offsets_are_bounds_checked(tmp_path):
    lib = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(S.__file__))), "lib",
                       "libsc23ad.so")
    shutil.copy(lib, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True,
                   capture_output=True)
    kernels, accesses, bad = set(), 0, set()
    for f in sorted(p for p in os.listdir(tmp_path) if p.endswith("gfx950")):
        dump = subprocess.Popen([OBJDUMP, "-d", "--no-show-raw-insn", f], cwd=tmp_path, text=True,
                                stdout=subprocess.PIPE)
        name = None
        for line in dump.stdout:
            if ANY.match(line):
                m = KERNEL.match(line)
                name = m.group(1) if m else None
                if name:
                    kernels.add(name)
            elif name and "buffer_" in line:
                m = ACCESS.match(line)
                if m is None:  # cache control has no operands
                    assert re.match(r"^\s+buffer_(inv|wbl2)", line), line
                    continue
                accesses += 1
                if m.group(2) != "0":
                    bad.add(name)
        assert dump.wait() == 0
    assert len(kernels) > 100 and accesses > 10 * len(kernels)
    assert not bad, f"{len(bad)} of {len(kernels)} kernels, first: {min(bad)}"
