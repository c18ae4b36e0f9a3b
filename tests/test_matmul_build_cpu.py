"""What the compiler says about the matrix kernels (csrc/matmul.hip), built for the device
with the Makefile's own flags: their inline asm is accepted without a warning (a register
clobber that the compiler does not honour would be one), and no register is spilled
where the code relies on it.
"""
import os
import shlex
import subprocess

import pytest
from helpers import ROOT

PKG = os.path.join(ROOT, "hbd-acestep.cpp_amd")


@pytest.fixture(scope="module")
def device_asm(tmp_path_factory):
    """(assembly, compiler messages) of csrc/matmul.hip."""
    lines = subprocess.run(["make", "-n", "-B", "-C", PKG], capture_output=True, text=True, check=True).stdout.splitlines()
    cmd = shlex.split(next(l for l in lines if " -c csrc/matmul.hip" in l))
    out = str(tmp_path_factory.mktemp("asm") / "matmul.s")
    cmd = cmd[:cmd.index("-c")] + ["--cuda-device-only", "-S", "csrc/matmul.hip", "-o", out]
    r = subprocess.run(cmd, cwd=PKG, capture_output=True, text=True, check=True)
    return open(out).read(), r.stderr


def test_inline_asm_compiles_without_warnings(device_asm):
    assert "inline-asm" not in device_asm[1], device_asm[1]


def test_kernels_that_count_their_loads_do_not_spill(device_asm):
    """The waits of the 64 x 64 kernel's pipeline count its loads in flight: a spill to memory
    among them would make every wait longer, with nothing else to show it."""
    meta = device_asm[0].split(".name: ")
    kernel = next(m for m in meta if m.strip().startswith("_ZN2mi12k_mmq64_q8_0"))
    assert ".vgpr_spill_count: 0" in kernel and ".private_segment_fixed_size: 0" in kernel, kernel[:1500]
