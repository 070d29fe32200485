"""Narrow outputs of the row-major GEMM where the K loop changes form (four steps at a time, the rest one by one): K at, one step
below and above whole turns of four and of sixteen waves, ends inside a fragment, rows and columns past the tile, strided rows,
rows that may not be read by whole fragments."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,pad,shift", [(1, 17, 240, 0, 0), (16, 40, 256, 8, 0), (16, 300, 272, 0, 0), (5, 33, 512, 0, 0), (17, 16, 1024, 8, 0),
                                             (40, 17, 2040, 0, 0), (16, 16, 2048, 0, 0), (300, 64, 2064, 8, 0), (2200, 17, 1000, 0, 0),
                                             (2100, 33, 4103, 1, 0), (16, 17, 512, 0, 1)])
def test_against_float64(dtype, M, N, K, pad, shift):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    rn = lambda r: torch.randn(r * (K + pad) + shift, generator=g, device="cuda").to(dtype)[shift:].view(r, K + pad)[:, :K]  # noqa: E731
    x, w = rn(M), rn(N)
    out = torch.full((M, N), float("nan"), device="cuda")
    ops.gemm_rm(x, w, out)
    ref = x.double() @ w.double().T.contiguous()
    # K products in fp32 sums: a walk of K roundings of 2^-24 of a partial sum, itself at most the root of K in size
    assert float((out.double() - ref).norm() / ref.norm()) <= 4 * K ** 0.5 * 2.0 ** -24
