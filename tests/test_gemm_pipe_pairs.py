"""Which workgroups of the 256 x 256 pipeline take two tiles (gemm_pipe.hip pairs_of): host code only."""
import heapq

import torch

from distributed_sse_for_llm_response_amd import ops


def _end(jobs, cus):
    """Every workgroup, in order, on the CU that is free first."""
    free = [0] * cus
    for j in jobs:
        heapq.heappush(free, heapq.heappop(free) + j)
    return max(free)


def test_held_cus_cost_what_they_do_without_pairs():
    ops.load_library(required=True)
    seen = 0
    for tiles in range(64, 4200, 61):
        pairs = torch.ops.dsse.gemm_pipe_pairs(tiles)
        assert 0 <= pairs and 512 * pairs <= tiles
        seen = max(seen, pairs)
        jobs = [2] * (256 * pairs) + [1] * (tiles - 512 * pairs)
        for held in (0, 8, 16, 32, 64):
            assert _end(jobs, 256 - held) <= _end([1] * tiles, 256 - held)
    assert seen >= 6
