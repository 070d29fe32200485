"""Which fp32 row-major products go to the tiles whose waves share K (host code only): both sides of the measured lines."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops


@pytest.mark.parametrize("M,N,K,batch,form", [
    (400, 2048, 2048, 1, 72), (400, 16384, 2048, 1, 0), (67, 32768, 2048, 1, 54), (400, 6272, 2048, 1, 54), (130, 16384, 2048, 1, 92), (300, 2048, 2048, 1, 52),
    (64, 8192, 2048, 1, 42), (40, 8192, 512, 1, 32), (113, 1030, 544, 4, 32),
    (100, 2048, 2048, 1, 0), (256, 1024, 512, 1, 0), (257, 1024, 512, 1, 32), (1500, 4096, 8192, 1, 0), (600, 16384, 2048, 1, 0),
    (64, 2048, 480, 1, 32), (512, 2048, 256, 1, 42), (520, 2048, 256, 1, 0), (64, 2048, 96, 1, 0), (300, 2048, 128, 1, 0)])
def test_form(M, N, K, batch, form):
    ops.load_library(required=True)
    assert torch.ops.dsse.gemm_rm_split_form(M, N, K, batch) == form
