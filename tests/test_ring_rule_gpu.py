"""Products of 17 to 64 rows on both sides of the lines where the ring takes eight waves instead of four and stops splitting K: one
round of workgroups of either kind, and widths that eight waves do not divide."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops import reference as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [17, 33, 64])
@pytest.mark.parametrize("N,K", [(8192, 512), (8256, 512), (10240, 1024), (16384, 512), (16448, 512), (16512, 512), (24448, 512), (4096, 4096)])
def test_products(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g, device="cuda") / K ** 0.5).to(torch.bfloat16)
    out = torch.full((M, N), float("nan"), device="cuda")
    ops.gemm_out(x, ref.tile_weight(w.cpu()).cuda(), out)
    want = x.double() @ w.double().T.contiguous()
    # exact products, fp32 sums: a random walk of K roundings of 2^-24 of a partial sum, four standard deviations
    assert float((out.double() - want).norm() / want.norm()) <= 4 * K ** 0.5 * 2.0 ** -24
