"""fp32 row-major products whose waves share a tile's K (gemm_rm_split.hip) against float64: every tile shape, rows and columns at the
tiles' edges, even and odd counts of chunks down to fewer than the stages, batches, slices of wider buffers, bias and activation."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops

pytestmark = pytest.mark.gpu


# rows one past, at and one short of a tile's; columns that end inside a tile's first and last 16
@pytest.mark.parametrize("M,N,K,Z,form", [
    (395, 6250, 544, 1, 54), (80, 32700, 512, 1, 54), (129, 16379, 512, 1, 92), (143, 16350, 544, 1, 92), (400, 2047, 544, 1, 72), (385, 2033, 512, 1, 72), (113, 1030, 544, 4, 32),
    (300, 2047, 512, 1, 52), (289, 2017, 544, 1, 52), (64, 8190, 544, 1, 42), (193, 2031, 2048, 1, 42), (33, 65, 160, 4, 32), (49, 2015, 128, 1, 32)])
def test_against_float64(M, N, K, Z, form):
    ops.load_library(required=True)
    assert torch.ops.dsse.gemm_rm_split_form(M, N, K, Z) == form
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(Z, M, K + 32, generator=g, device="cuda")[:, :, :K]
    w = (torch.randn(Z, N, K + 64, generator=g, device="cuda") / K ** 0.5)[:, :, 32:K + 32]
    bias = torch.randn(Z, N, generator=g, device="cuda")
    if Z == 1:
        x, w, bias = x[0], w[0], bias[0]
    x[..., M // 2, K // 2] = float("inf")  # one row's results alone
    ref = x.double() @ w.double().transpose(-1, -2).contiguous()
    # fp32 sums of K rounded products: a random walk of K steps of at most 2^-24 of the partial sum, four standard deviations
    bound = 4.0 * (K + 1) ** 0.5 * 2.0 ** -24
    rest = [i for i in range(M) if i != M // 2]
    for b, act in ((None, 0), (bias, 0), (bias, 1)):
        want = ref if b is None else ref + b.double().unsqueeze(-2)
        if act:
            want = torch.nn.functional.gelu(want, approximate="tanh")
        wide = torch.full((*ref.shape[:-1], N + 3), float("nan"), device="cuda")
        out = wide[..., :N]
        ops.gemm_rm(x, w, out, bias=b, act=act)
        assert float((out[..., rest, :].double() - want[..., rest, :]).norm() / want[..., rest, :].norm()) <= bound
        assert not torch.isfinite(out[..., M // 2, :]).all() and torch.isnan(wide[..., N:]).all()
