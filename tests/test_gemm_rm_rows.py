"""Which form an fp32 row-major product of many tiles takes (host code only): the rows of a tile that were measured to be through first,
on both sides of the lines: third rounds nearly empty and full, one round, a second of few workgroups, batches."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops


@pytest.mark.parametrize("M,N,batch,rows", [
    (330, 8192, 1, 48), (200, 12288, 1, 48), (240, 12288, 1, 48), (330, 16384, 1, 48), (80, 12288, 1, 48), (560, 12288, 1, 48),
    (400, 8192, 1, 64), (480, 8192, 1, 64), (200, 16384, 1, 64), (300, 12288, 1, 64), (560, 6272, 1, 64), (240, 16384, 1, 64),
    (130, 16384, 1, 80), (400, 6272, 1, 80), (400, 16384, 1, 80), (560, 4096, 1, 80), (640, 8192, 1, 80),
    (330, 2048, 1, 48), (400, 2048, 1, 64), (330, 2048, 4, 48), (3000, 16384, 1, 64)])
def test_form(M, N, batch, rows):
    ops.load_library(required=True)
    assert torch.ops.dsse.gemm_rm_form_rows(M, N, batch) == rows
