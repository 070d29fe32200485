"""The GEMM tile that holds all of 65 to 256 rows (gemm_tiled cfg 2): its plan (host code) and its products."""
import math

import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops import reference as R


# one round of workgroups at most, wide products from 129 rows on, slices only where they were measured to pay
@pytest.mark.parametrize("M,N,K,slabs,want", [
    (64, 28672, 4096, False, None), (65, 28672, 4096, False, 1), (192, 28672, 4096, False, 1), (224, 28672, 4096, False, 1), (225, 28672, 4096, False, None),
    (160, 32768, 4096, False, 1), (160, 32896, 4096, False, None), (128, 26752, 4096, False, None), (129, 14464, 4096, False, 2),
    (256, 26752, 4096, False, 1), (257, 26752, 4096, False, None), (160, 14464, 2048, False, 1), (72, 8320, 2048, False, 2),
    (72, 10368, 4096, False, None), (160, 12288, 2048, False, None), (160, 14464, 1536, False, 1), (208, 14336, 2048, False, None), (128, 28672, 4096, False, None),
    (96, 28672, 4096, False, 1), (128, 32768, 2048, False, 1), (200, 10240, 4096, False, None), (200, 16384, 4096, False, 2), (160, 8192, 4096, False, None),
    (160, 6144, 4096, True, None), (160, 8192, 4096, True, 4), (160, 4096, 14336, True, 8), (160, 2048, 8192, True, None), (160, 4096, 4096, True, None), (200, 4096, 14336, True, None)])
def test_plan(M, N, K, slabs, want):
    ops.load_library(required=True)
    impl, cfg, split, fix, _ = torch.ops.dsse.gemm_plan(M, N, K, slabs)
    assert ((impl, cfg) == (4, 2)) == (want is not None)
    if want is not None:
        assert (split, fix) == (want, False)


# a key that shapes another kernel means that kernel: the size rules step aside, here and in the rules of fewer rows
@pytest.mark.parametrize("M,N,K,key,value,want", [
    (160, 14464, 4096, "t_split", 1, (3, -1, 0)), (72, 32768, 4096, "w_split", 1, (3, -1, 0)), (72, 32768, 4096, "w_rd", 2, (3, -1, 0)),
    (72, 8320, 2048, "s_split", 2, (2, -1, 0)), (200, 16384, 4096, "t_fix", 1, (4, 5, 2)), (200, 16384, 4096, "t_small", 0, (4, 5, 2)),
    (16, 16384, 4096, "s_split", 1, (2, -1, 0)), (32, 2048, 2048, "s_ring", 1, (2, -1, 0)), (32, 2048, 2048, "resid_split", 4, (2, -1, 0)),
    (160, 16384, 4096, "t_split", 1, (4, 5, 1)), (160, 14464, 4096, "attn_pd", 1, (4, 2, 2))])
def test_plan_under_keys(monkeypatch, M, N, K, key, value, want):
    ops.load_library(required=True)
    monkeypatch.setenv("DSSE_KERNEL_CFG", ops.kernel_cfg_env(**{key: value}))
    ops.refresh_env()
    try:
        got = torch.ops.dsse.gemm_plan(M, N, K)[:3]
    finally:
        monkeypatch.undo()
        ops.refresh_env()
    assert got == want
    assert torch.ops.dsse.gemm_plan(M, N, K)[:3] != want or key == "attn_pd"


@pytest.fixture
def forced(monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    ops.load_library(required=True)

    def set_(S):
        monkeypatch.setenv("DSSE_KERNEL_CFG", ops.kernel_cfg_env(gemm_impl=4, t_cfg=2, t_split=S))
        ops.refresh_env()
    yield set_
    monkeypatch.undo()
    ops.refresh_env()


# both sides of every height, fewer K steps than stages, slices, several column blocks
@pytest.mark.gpu
@pytest.mark.parametrize("M", [65, 96, 97, 128, 129, 160, 161, 192, 193, 224, 225, 255, 256])
@pytest.mark.parametrize("N,K,S", [(128, 128, 1), (384, 384, 1), (256, 1024, 2)])
def test_products(forced, M, N, K, S):
    forced(S)
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    # rows past M would show: the buffer goes on with other values
    x = torch.randn(M + 40, K, device=dev, generator=g).bfloat16()[:M]
    w = R.tile_weight((torch.randn(N, K, device=dev, generator=g) / math.sqrt(K)).bfloat16())
    assert torch.ops.dsse.gemm_plan(M, N, K)[:3] == (4, 2, S)
    ref = x.double() @ R.untile_weight(w).double().t()
    big = float(ref.abs().max())
    f32 = torch.full((M, N), float("nan"), device=dev)
    ops.gemm_out(x, w, f32)
    assert float((f32 - ref).abs().max()) <= K * 2.0 ** -23 * big  # K fp32 additions
    bf = torch.full((M, N), float("nan"), device=dev, dtype=torch.bfloat16)
    ops.gemm_out(x, w, bf)
    assert float((bf - ref).abs().max()) <= 2.0 ** -8 * big
    resid = torch.randn(M, N, device=dev, generator=g)
    want = resid.double() + ref
    ops.gemm_resid(x, w, resid)
    assert float((resid - want).abs().max()) <= K * 2.0 ** -23 * big + 2.0 ** -21
    part = torch.full((S * M * N,), float("nan"), device=dev)
    if S > 1:
        assert ops.gemm_out_split(x, w, bf, part) == S
        assert float((part.view(S, M, N).sum(0) - ref).abs().max()) <= K * 2.0 ** -23 * big
    silu = torch.full((M, N // 2), float("nan"), device=dev, dtype=torch.bfloat16)
    ops.gemm_silu(x, w, silu)
    gu = ref.view(M, N // 16, 16)
    want = (torch.nn.functional.silu(gu[..., :8]) * gu[..., 8:]).reshape(M, N // 2)
    assert float((silu - want).abs().max()) <= 2.0 ** -8 * float(want.abs().max()) + K * 2.0 ** -22 * big * big
