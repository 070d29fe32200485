"""The 256 x 256 pipeline from two rounds of 256 tiles on, from three on with workgroups that go on to a second tile: the fewest K steps that they take, one more
and an odd count, a last round of a few tiles, ragged rows, a half-empty last column block, every tile height; results that are not aligned to 16 bytes."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops import reference as R

pytestmark = pytest.mark.gpu


@pytest.fixture
def tile(monkeypatch):
    def choose(cfg):
        monkeypatch.setenv("DSSE_KERNEL_CFG", ops.kernel_cfg_env(t_cfg=cfg, t_split=1 if cfg else None))
        ops.refresh_env()
    yield choose
    monkeypatch.undo()
    ops.refresh_env()


# tiles of 256 / 192 / 128 rows x 256 columns: 513, 531, 989, 533 and 561 of them, the half-empty column block as it is planned; and 774, 801, 780, 825 and 1287:
# one round of pairs and two
@pytest.mark.parametrize("cfg,M,N,K", [
    ("8", 2050, 14592, 256), ("8", 2300, 15104, 384), ("9", 8200, 5888, 256), ("10", 1537, 10496, 640), (None, 4200, 8320, 2048),
    ("8", 2050, 22016, 256), ("8", 2300, 22784, 384), ("10", 1537, 15360, 640), (None, 6200, 8320, 2048), ("8", 2050, 36608, 384)])
@pytest.mark.parametrize("shift", [0, 1])
def test_rounds(gpu, tile, cfg, M, N, K, shift):
    tile(cfg)
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).bfloat16()
    w = (torch.randn(N, K, generator=g) / K ** 0.5).bfloat16()
    wt, xc = R.tile_weight(w).to(gpu), x.to(gpu)
    want = (xc.float() @ w.to(gpu).float().t())
    empty = lambda n: torch.full((M * n + 8,), float("nan"), dtype=torch.bfloat16, device=gpu)  # noqa: E731
    buf = empty(N)
    out = buf[shift:shift + M * N].view(M, N)
    ops.gemm_out(xc, wt, out)
    # one rounding to bf16, 2^-9 of the value, beside fp32 sums of K products of about one
    torch.testing.assert_close(out.float(), want, rtol=2 ** -8, atol=2 ** -16 * K ** 0.5)
    assert torch.isnan(buf[:shift]).all() and torch.isnan(buf[shift + M * N:]).all()
    pairs = want.view(M, N // 16, 16)
    for fn, act in ((ops.gemm_silu, torch.nn.functional.silu), (ops.gemm_gelu, lambda z: torch.nn.functional.gelu(z, approximate="tanh"))):
        buf = empty(N // 2)
        out = buf[shift:shift + M * N // 2].view(M, N // 2)
        fn(xc, wt, out)
        ref = (act(pairs[..., :8]) * pairs[..., 8:]).reshape(M, N // 2)
        # as above, and the fast exponential's 2^-21 or so in the gate, which is up to some five times the product's scale
        torch.testing.assert_close(out.float(), ref, rtol=2 ** -8, atol=2 ** -14 * K ** 0.5)
        assert torch.isnan(buf[:shift]).all() and torch.isnan(buf[shift + M * N // 2:]).all()
