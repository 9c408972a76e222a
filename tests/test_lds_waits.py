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


def test_sums_of_squares_are_in_lds_before_a_barrier():
    """All waves write sums that one wave adds, and one wave what all read: nothing else orders them where a workgroup's first unit
    has a single chunk."""
    with open(os.path.join(CSRC, "gemm_bf16.hip")) as f:
        source = f.read()
    for write in (r"sq\[tid\] = t;", r"rstd\[lane\] = [^;]*;"):
        after = re.findall(write + r"\s*([^;]*);", source)
        assert len(after) == 1 and "s_waitcnt lgkmcnt(0)" in after[0], after


def test_statements_that_write_m0_say_so():
    """A statement that writes m0 without naming it lets the compiler keep a value of its own there."""
    for name in sorted(os.listdir(CSRC)):
        if not name.endswith((".hip", ".h")):
            continue
        with open(os.path.join(CSRC, name)) as f:
            statements = re.findall(r'asm volatile\((.*?)\);', f.read().replace("\\\n", "\n"), re.S)
        for text in statements:
            if re.search(r"\bm0\b", text.split("::")[0]):
                assert re.search(r':\s*[^:]*"m0"[^:]*$', text), (name, text)
