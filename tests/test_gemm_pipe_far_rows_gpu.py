"""fp32 results of the 256-row pipeline whose rows are megabytes apart: a tile's last rows lie more than 2 GiB behind its first one."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops import reference as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [4300032, 8388352])  # the second: the most columns whose weight fits the operator's 2 GiB
def test_far_rows(gpu, monkeypatch, N):
    monkeypatch.setenv("DSSE_KERNEL_CFG", ops.kernel_cfg_env(t_cfg=8, t_split=1))
    ops.refresh_env()
    try:
        M, K = 130, 128
        g = torch.Generator(device=gpu).manual_seed(N)
        x = torch.randn(M, K, generator=g, device=gpu).bfloat16()
        w = torch.randn(N, K, generator=g, device=gpu).bfloat16()
        wt = R.tile_weight(w)
        out = torch.full((M, N), float("nan"), device=gpu)
        ops.gemm_out(x, wt, out)
        rows = [0, 63, 64, 65, 124, 125, 126, 127, 128, 129]
        # fp32 sums of 128 products of about one
        torch.testing.assert_close(out[rows], x[rows].float() @ w.float().t(), rtol=2 ** -16, atol=2 ** -14)
        assert not torch.isnan(out).any()
    finally:
        monkeypatch.undo()
        ops.refresh_env()
        torch.cuda.empty_cache()
