"""Rings in LDS that direct loads fill: the wait before a stage is asked for again is also one for the reads of what it held, in
the source and not by the place that the compiler happens to give the instructions that use them."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "braidinfer_amd", "csrc")


@pytest.mark.parametrize("source,waits", [("gemm_f32.hip", 2), ("routed_experts.hip", 2)])
def test_waits_for_loads_are_waits_for_reads(source, waits):
    with open(os.path.join(CSRC, source)) as f:
        found = re.findall(r'asm volatile\("s_waitcnt (vmcnt\([^"]*)"', f.read())
    assert len(found) == waits and all("lgkmcnt(0)" in w for w in found), found
