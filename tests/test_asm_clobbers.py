"""Inline assembly of the kernels that writes m0 says so: the compiler keeps no value of its own there."""
import glob
import os
import re

from hydra_amd import build


def test_assembly_that_writes_m0_declares_it():
    seen = 0
    for path in sorted(glob.glob(os.path.join(build.CSRC, "*.h*"))):
        for stmt in re.findall(r"asm volatile\((.*?)\);", open(path).read(), flags=re.S):
            if re.search(r"s_mov_b32\s+m0\b", stmt):
                seen += 1
                assert '"m0"' in stmt.rsplit(":", 1)[-1], (path, stmt)   # the clobbers come last
    assert seen
