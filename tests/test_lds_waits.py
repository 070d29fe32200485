"""GEMM rings that refill the LDS slot of the step before right after a step's barrier: the barrier itself waits for the wave's LDS reads,
wherever the compiler puts their wait."""
import re
from pathlib import Path

import pytest

KERNELS = Path(__file__).resolve().parent.parent / "csrc" / "kernels"
WAIT = re.compile(r'asm volatile\("s_waitcnt (vmcnt\([^"]*?)\\n\\ts_barrier" ::([^;]*);')


# the barriers of each file that compute waves reach; the X loader of gemm_stream.hip's decoupled ring reads no LDS
@pytest.mark.parametrize("name,barriers,without_reads", [
    ("gemm_tiled.hip", 3, ()), ("gemm_rowmajor.hip", 2, ()), ("gemm_stream.hip", 3, ('"n"((DX - 2) * XI)',))])
def test_barrier_waits_for_reads(name, barriers, without_reads):
    found = WAIT.findall((KERNELS / name).read_text())
    assert len(found) == barriers
    for wait, operands in found:
        if not any(x in operands for x in without_reads):
            assert "lgkmcnt(0)" in wait, (wait, operands)
