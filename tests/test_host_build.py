"""What the host code of the library asks of the processor: x86-64 alone, except for the second build of the
edge collapse, which is taken only where the processor counts bits in hardware."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "specseqplusplus_amd", "csrc")


@pytest.mark.skipif(shutil.which("make") is None, reason="no make")
def test_only_the_second_collapse_asks_for_an_instruction():
    out = subprocess.run(["make", "-n", "-B", "-C", CSRC, "all"], capture_output=True, text=True, check=True).stdout
    compiles = [line.split() for line in out.splitlines() if " -o " in line]
    asking = [c for c in compiles if any(w.startswith("-m") for w in c)]
    assert len(compiles) > 8 and len(asking) == 1
    assert "ssq_collapse.cpp" in asking[0] and "-DSSQ_COLLAPSE_POPCNT" in asking[0]
    assert [w for w in asking[0] if w.startswith("-m")] == ["-mpopcnt"]
