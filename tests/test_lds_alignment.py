"""The kernels that find LDS pieces by XOR of address bits 4 to 6 (the element records of
the block pass, the block records of the two-sided scaling) declare their arrays at
multiples of 128 bytes, and the 16-byte operand reads of the weight gradient theirs at 16:
the alignment the compiler's front end gives each LDS array, from the sources."""
import os
import re
import shutil
import subprocess

import pytest

from phasta_amd import build

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
pytestmark = pytest.mark.skipif(shutil.which(HIPCC) is None, reason="needs hipcc")


@pytest.mark.parametrize("source,arrays,align", [
    ("k_assembly.hip", r"(asm_pairs|k_asm_blocks).*E3lds$", 128),
    ("k_solver.hip", r"k_spsi3pre.*E7lds_all$", 128),
    ("k_mpnn.hip", r"k_mp_dW.*E2s[AU]$", 16),
])
def test_declared_alignment(source, arrays, align, tmp_path):
    out = tmp_path / "module.ll"
    subprocess.run([HIPCC, *build.HIPCC_FLAGS[:1], "-std=c++17", f"-I{build.INC}", "-O1",
                    "-Xclang", "-disable-llvm-passes", "--cuda-device-only", "-S", "-emit-llvm",
                    os.path.join(build.CSRC, source), "-o", str(out)],
                   check=True, stderr=subprocess.DEVNULL)
    found = re.findall(r"^@(\S+) = .*addrspace\(3\) global .*, align (\d+)$", out.read_text(),
                       re.MULTILINE)
    mine = [(n, int(a)) for n, a in found if re.search(arrays, n)]
    assert mine
    assert all(a >= align for _, a in mine), mine
