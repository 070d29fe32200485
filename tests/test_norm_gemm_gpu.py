"""Products of RMS-normalised fp32 rows in one launch against the norm and the product apart: the smallest and largest row counts and
widths that the launch takes, waves that have no second chunk, and what it refuses."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
EPS = 1e-5


def _operands(M, N, K):
    g = torch.Generator().manual_seed(M + N + K)
    resid = torch.randn(M, K, generator=g) * 3
    nw = (1 + 0.2 * torch.randn(K, generator=g)).to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16)
    wt = ref.tile_weight(w)
    return resid, nw, wt


@pytest.mark.parametrize("M,N,K", [(1, 16, 1024), (4, 48, 1024), (3, 32, 2048), (2, 256, 3072), (1, 160, 4096), (4, 6144, 4096),
                                   (1, 64, 6144), (2, 32, 8192)])
def test_normalised_products(M, N, K):
    assert ops.norm_gemm_ok(M, N, K)
    resid, nw, wt = _operands(M, N, K)
    c = lambda t: t.cuda()  # noqa: E731
    x = torch.empty(M, K, dtype=torch.bfloat16, device="cuda")
    ops.rmsnorm(c(resid), c(nw), x, EPS)
    # the sums of squares are taken in another order: a normalised value may round to its bf16 neighbour (2^-8 of it), one product
    # of K unit-variance terms over sqrt(K) weights then moves by 2^-8 / sqrt(K) of a typical output each: 3 * 2^-8 covers all of them
    tol = dict(atol=3 * 2 ** -8, rtol=2 ** -7)
    two, one = (torch.empty(M, N, device="cuda") for _ in range(2))
    ops.gemm_out(x, c(wt), two)
    ops.norm_gemm_out(c(resid), c(nw), EPS, c(wt), one)
    torch.testing.assert_close(one, two, **tol)
    want = torch.empty(M, N)
    ref.gemm_out(ref.normed(resid, nw, EPS), wt, want)
    torch.testing.assert_close(one.cpu(), want, **tol)
    two, one = (torch.empty(M, N // 2, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    ops.gemm_silu(x, c(wt), two)
    ops.norm_gemm_silu(c(resid), c(nw), EPS, c(wt), one)
    torch.testing.assert_close(one.float(), two.float(), atol=2 ** -5, rtol=2 ** -6)


@pytest.mark.parametrize("M", [1, 3])
def test_normalised_qkv(M):
    nh, nkv, K, blocks = 8, 2, 4096, 6
    resid, nw, wt = _operands(M, (nh + 2 * nkv) * 128, K)
    c = lambda t: t.cuda()  # noqa: E731
    pos, slots = torch.tensor([5, 40, 2][:M], dtype=torch.int32), torch.tensor([37, -1, 100][:M], dtype=torch.int32)
    rope = torch.randn(64, 64, 2, generator=torch.Generator().manual_seed(1))
    x = torch.empty(M, K, dtype=torch.bfloat16, device="cuda")
    ops.rmsnorm(c(resid), c(nw), x, EPS)
    out = []
    for norm in (False, True):
        q = torch.zeros(M, nh * 128, dtype=torch.bfloat16, device="cuda")
        kc = torch.zeros(blocks, nkv, 32, 128, dtype=torch.bfloat16, device="cuda")
        vc = torch.zeros(blocks, nkv, 128, 32, dtype=torch.bfloat16, device="cuda")
        rest = (c(wt), c(pos), c(slots), c(rope), q, kc, vc, nh, nkv)
        ops.norm_gemm_qkv_rope(c(resid), c(nw), EPS, *rest) if norm else ops.gemm_qkv_rope(x, *rest)
        out.append((q, kc, vc))
    for a, b in zip(*out):
        torch.testing.assert_close(a.float(), b.float(), atol=2 ** -5, rtol=2 ** -6)


def test_refused():
    resid, nw, wt = _operands(5, 64, 1024)
    for M, N, K in ((5, 64, 1024), (3, 64, 8192), (0, 64, 1024), (1, 60, 1024), (1, 64, 512), (1, 64, 5120), (1, 64, 1088), (1, 64, 16384)):
        assert not ops.norm_gemm_ok(M, N, K)
    with pytest.raises(RuntimeError):
        ops.norm_gemm_out(resid.cuda(), nw.cuda(), EPS, wt.cuda(), torch.empty(5, 64, device="cuda"))
