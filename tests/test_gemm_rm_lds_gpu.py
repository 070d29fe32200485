"""The LDS-staged forms of the general row-major GEMM (gemm_rowmajor.hip) against float64, at the edges of their tiles,
chunks and wave groups."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    ops.load_library(required=True)
    return torch.device("cuda", 0)


def check(out, ref, K):
    """fp32 sums of K exact (bf16) or rounded (fp32) products: rounding errors add up like a random walk of K steps, each at
    most 2^-24 of the partial sum, four standard deviations allowed; a bf16 result is rounded once more, by 2^-9 at most."""
    bound = 4.0 * (K + 1) ** 0.5 * 2.0 ** -24 + (2.0 ** -9 if out.dtype == torch.bfloat16 else 0.0)
    err = float((out.double() - ref).norm() / ref.norm())
    assert err <= bound, (err, bound)


# M, N, chunks of 128 bytes per row, batch: 32 x 32 tiles with four wave groups (chunk counts below, at and above a multiple
# of four, tile edges on both sides), 64 x 64 tiles with two groups (odd and even counts of chunks), with one group (batches
# and more tiles than CUs), and a count that leaves a group without a chunk
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,chunks,Z", [
    (17, 65, 1, 1), (31, 96, 2, 1), (32, 100, 3, 1), (33, 129, 5, 2), (64, 255, 8, 1), (65, 320, 17, 1), (1000, 520, 9, 1),
    (700, 1000, 8, 1), (63, 100, 4, 70), (257, 2050, 3, 2), (1100, 1024, 1, 1), (1030, 1100, 2, 3), (1030, 1100, 4, 1)])
def test_against_float64(gpu, dtype, M, N, chunks, Z):
    K = chunks * 128 // torch.empty(0, dtype=dtype).element_size()
    g = torch.Generator(device=gpu).manual_seed(M + N + chunks)
    # operands and result are slices of wider buffers: rows further apart than their length
    x = torch.randn(Z, M, K + 32, generator=g, device=gpu).to(dtype)[:, :, :K]
    w = (torch.randn(Z, N, K + 64, generator=g, device=gpu) / K ** 0.5).to(dtype)[:, :, 32:K + 32]
    bias = torch.randn(Z, N, generator=g, device=gpu).to(dtype)
    if Z == 1:
        x, w, bias = x[0], w[0], bias[0]
    ref = x.double() @ w.double().transpose(-1, -2).contiguous()
    for out_t in {torch.float32, dtype}:
        wide = torch.full((*ref.shape[:-1], N + 3), float("nan"), device=gpu, dtype=out_t)
        ops.gemm_rm(x, w, wide[..., :N])
        check(wide[..., :N], ref, K)
        assert torch.isnan(wide[..., N:]).all()
        ops.gemm_rm(x, w, wide[..., :N], bias=bias)
        check(wide[..., :N], ref + bias.double().unsqueeze(-2), K)
