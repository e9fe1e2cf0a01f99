"""Dynamic LDS is read as 16-byte vectors (knots, beads, frames), so it has to begin on 16 bytes.

It begins behind a kernel's own ``__shared__`` data, whose size follows the kernel's code: an array
of doubles declared as it is begins 8 bytes off behind an odd number of them.  Every kernel's
declaration therefore asks for the alignment, which also rounds the size that the compiler notes for
the kernel's own data.
"""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "moribs-pimc_amd", "csrc")
ALIGNED = ("uint4", "float4", "double2", "double4")  # types whose own alignment is 16 bytes or more


@pytest.mark.parametrize("path", sorted(glob.glob(os.path.join(CSRC, "*.h*"))), ids=os.path.basename)
def test_dynamic_lds_begins_on_16_bytes(path):
    with open(path) as f:
        src = f.read()
    for line in re.findall(r"extern __shared__[^;]*;", src):
        typ = re.search(r"(\w+)\s+\w+\[\];", line).group(1)
        assert "DYNAMIC_LDS" in line or "alignas(16)" in line or typ in ALIGNED, line
    if "DYNAMIC_LDS" in src:
        assert re.search(r"#define DYNAMIC_LDS __attribute__\(\(aligned\(16\)\)\)", src)
