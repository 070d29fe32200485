"""Which tiled-layout GEMM a product with a half-empty last column block (N % 256 == 128) is planned for: host code only."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops


def plan(M, N, K):
    ops.load_library(required=True)
    impl, cfg, split, fix, _ = torch.ops.dsse.gemm_plan(M, N, K, False)
    return impl, cfg >= 8, split, fix


# measured faster in 128-column tiles: short reductions in one full round of them, few long rounds against slices of up to 2048
@pytest.mark.parametrize("M,N,K", [(1800, 3200, 512), (1100, 5248, 512), (1500, 26752, 4096), (2500, 14464, 4096), (600, 26752, 8192),
                                   (700, 26752, 8192), (6000, 3200, 8192)])
def test_narrow_tiles(M, N, K):
    assert plan(M, N, K) == (4, False, 1, False)


# measured faster on the 256-column pipeline, combined in the launch or not
@pytest.mark.parametrize("M,N,K", [(1800, 8320, 4096), (1100, 14464, 4096), (2500, 14464, 8192), (2500, 26752, 8192), (1500, 26752, 8192),
                                   (2048, 26752, 4096), (257, 8320, 2048), (1500, 1152, 2048), (3000, 1152, 512)])
def test_pipeline(M, N, K):
    impl, pipe, _, _ = plan(M, N, K)
    assert impl == 4 and pipe
