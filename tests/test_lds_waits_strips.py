"""The fp32 strips and expert GEMMs refill the slot of the chunk before right after a chunk's barrier, as the kernels of
test_lds_waits.py do: their barriers wait for the wave's LDS reads too."""
import pytest
from test_lds_waits import test_barrier_waits_for_reads as waits


@pytest.mark.parametrize("name", ["gemm_rm_strip.hip"])
def test_counted(name):
    waits(name, 1, ())


def test_fixed_count():
    from test_lds_waits import KERNELS

    text = (KERNELS / "moe_exact.hip").read_text()
    assert text.count("s_barrier") == 1 and 's_waitcnt vmcnt(8) lgkmcnt(0)\\n\\ts_barrier"' in text
