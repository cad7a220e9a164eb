"""Registers of the built kernels (no GPU needed): a register too many costs a
wave per SIMD, and a small change elsewhere can bring one, so the counts that
the kernels' occupancy rests on are read from the library's own metadata."""
import os
import re
import shutil
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "beedrill_amd",
                   "libbeedrill_amd.so")
LLVM = "/opt/rocm/llvm/bin"

pytestmark = pytest.mark.skipif(not os.path.exists(os.path.join(LLVM, "llvm-objdump")),
                                reason="no LLVM tools to read the library with")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    d = tmp_path_factory.mktemp("objects")
    lib = shutil.copy(LIB, d / "lib.so")
    subprocess.run([os.path.join(LLVM, "llvm-objdump"), "--offloading", lib], check=True, cwd=d,
                   capture_output=True)
    out = {}
    for f in d.glob("lib.so.*gfx950"):
        notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", str(f)], check=True,
                               capture_output=True, text=True).stdout
        for name, vgprs, spills in re.findall(
                r"\.name: +(\S+)\n(?:(?!\.name:).)*?\.vgpr_count: +(\d+)\n +\.vgpr_spill_count: (\d+)",
                notes, re.S):
            out[name] = int(vgprs), int(spills)
    return out


@pytest.mark.parametrize("name,number,registers", [
    ("k_step", 9, 96),     # five waves a SIMD
    ("k_cc_hook", 2, 64),  # eight
    ("k_solo", 1, 128),    # four: one workgroup of 16 waves
])
def test_registers(kernels, name, number, registers):
    found = {k: v for k, v in kernels.items() if re.search(r"\d+%s(?=[IE])" % name, k)}
    assert len(found) == number, sorted(found)
    for k, (vgprs, spills) in found.items():
        assert vgprs <= registers and spills == 0, (k, vgprs, spills)
