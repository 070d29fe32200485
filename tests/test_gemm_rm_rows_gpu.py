"""fp32 row-major products in strips of 48 and 80 rows against float64: rows and columns at the strips' edges, one chunk more and fewer
than the stages, batches, slices of wider buffers; results do not depend on the form, so rows of one product agree with those of a
product of fewer rows that takes another."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops

pytestmark = pytest.mark.gpu


def _bound(K):
    """fp32 sums of K rounded products: a random walk of K steps of at most 2^-24 of the partial sum, four standard deviations."""
    return 4.0 * (K + 1) ** 0.5 * 2.0 ** -24


# (48-row strips: 130, 81, 240 and 800 rows; 80-row strips: 400 and 330; 64 x 64: 97 and 256) x columns that end inside a strip's 64
@pytest.mark.parametrize("M,N,K,Z", [(130, 8200, 96, 1), (97, 16390, 128, 1), (400, 6272, 160, 1), (330, 2051, 96, 3), (400, 16384, 32, 1),
                                     (81, 16300, 256, 1), (256, 8192, 96, 1), (240, 12000, 2048, 1), (800, 3300, 544, 1)])
def test_strips(M, N, K, Z):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(Z, M, K + 32, generator=g, device="cuda")[:, :, :K]
    w = (torch.randn(Z, N, K + 64, generator=g, device="cuda") / K ** 0.5)[:, :, 32:K + 32]
    bias = torch.randn(Z, N, generator=g, device="cuda")
    if Z == 1:
        x, w, bias = x[0], w[0], bias[0]
    ref = x.double() @ w.double().transpose(-1, -2).contiguous()
    wide = torch.full((*ref.shape[:-1], N + 3), float("nan"), device="cuda")
    ops.gemm_rm(x, w, wide[..., :N])
    assert float((wide[..., :N].double() - ref).norm() / ref.norm()) <= _bound(K)
    assert torch.isnan(wide[..., N:]).all()
    part = torch.empty(*ref.shape[:-2], 64, N, device="cuda")
    ops.gemm_rm(x[..., :64, :], w, part)
    assert float((part - wide[..., :64, :N]).abs().max()) <= _bound(K) * 40
    ops.gemm_rm(x, w, wide[..., :N], bias=bias)
    ref += bias.double().unsqueeze(-2)
    assert float((wide[..., :N].double() - ref).norm() / ref.norm()) <= _bound(K)
