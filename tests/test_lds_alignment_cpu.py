"""Dynamic LDS arrays start after a kernel's static ones, at an address that only the
array's own alignment fixes: one of bytes has to declare the alignment of the widest
access made through it (16 bytes).
"""
import glob
import os
import re

from helpers import ROOT


def test_dynamic_lds_arrays_declare_their_alignment():
    decl = re.compile(r"extern\s+__shared__\s+([^;]*);")
    found = 0
    for path in glob.glob(os.path.join(ROOT, "hbd-acestep.cpp_amd", "csrc", "*.hip")):
        for d in decl.findall(open(path).read()):
            found += 1
            if re.match(r"(__attribute__\S+\s+)?char\b", d):
                assert "aligned(16)" in d, f"{os.path.basename(path)}: extern __shared__ {d}"
    assert found
