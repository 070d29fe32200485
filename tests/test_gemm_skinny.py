"""Which products of up to 64 rows the skinny GEMM takes (host code), and those products."""
import math

import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops import reference as R


# wide outputs of 9 to 16 rows in full or well filled rounds of two-tile workgroups; narrow, short products of 17 to 64 rows
@pytest.mark.parametrize("M,N,K,skinny", [
    (16, 16384, 4096, True), (16, 32768, 2048, True), (16, 26752, 4096, False), (16, 28672, 4096, False), (9, 10240, 4096, True),
    (17, 4096, 2048, True), (17, 4224, 2048, False), (32, 2048, 2560, True), (32, 2048, 3072, False), (32, 4096, 1792, False), (33, 2048, 2048, False),
    (64, 2048, 1024, True), (64, 2048, 1536, False)])
def test_plan(M, N, K, skinny):
    ops.load_library(required=True)
    assert (torch.ops.dsse.gemm_plan(M, N, K)[0] == 0) == skinny


# the same products where the next kernel sums the slices (a tensor-parallel shard's o projection before its norm): sliced
@pytest.mark.parametrize("M,N,K", [(17, 4096, 2048), (32, 2048, 2560), (64, 2048, 1024), (32, 4096, 512)])
def test_plan_before_a_slab_consumer(M, N, K):
    ops.load_library(required=True)
    assert torch.ops.dsse.gemm_plan(M, N, K)[0] == 0
    assert torch.ops.dsse.gemm_plan(M, N, K, True)[0] == 2


# and those calls leave slabs: their sum is the product
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(17, 4096, 2048), (64, 2048, 1024)])
def test_slabs(M, N, K):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    ops.load_library(required=True)
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    w = R.tile_weight((torch.randn(N, K, device="cuda", generator=g) / math.sqrt(K)).bfloat16())
    ref = x.double() @ R.untile_weight(w).double().t()
    for call, out in ((ops.gemm_out_split, torch.zeros(M, N, device="cuda", dtype=torch.bfloat16)), (ops.gemm_resid_split, torch.zeros(M, N, device="cuda"))):
        part = torch.full((16 * M * N,), float("nan"), device="cuda")
        S = call(x, w, out, part)
        assert S > 1
        assert float((part[:S * M * N].view(S, M, N).sum(0) - ref).abs().max()) <= K * 2.0 ** -23 * float(ref.abs().max())  # K fp32 additions


# both sides of two column tiles per wave (8 and 16 rows, full and nearly empty last rounds), the first and last row of a 16-row
# tile in the 32- and 64-row forms, K walks shorter than the waves that share them
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(7, 5120, 256), (8, 5120, 128), (16, 5120, 384), (15, 8192, 1152), (16, 8320, 256), (17, 256, 512),
                                   (32, 4096, 1536), (31, 128, 2560), (33, 256, 1024), (64, 128, 512)])
def test_products(M, N, K):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    ops.load_library(required=True)
    assert torch.ops.dsse.gemm_plan(M, N, K)[0] == 0
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn(M, K, device=dev, generator=g).bfloat16()
    w = R.tile_weight((torch.randn(N, K, device=dev, generator=g) / math.sqrt(K)).bfloat16())
    ref = x.double() @ R.untile_weight(w).double().t()
    big = float(ref.abs().max())
    out = torch.full((M, N), float("nan"), device=dev)
    ops.gemm_out(x, w, out)
    assert float((out - ref).abs().max()) <= K * 2.0 ** -23 * big  # K fp32 additions
    resid = torch.randn(M, N, device=dev, generator=g)
    want = resid.double() + ref
    ops.gemm_resid(x, w, resid)
    assert float((resid - want).abs().max()) <= K * 2.0 ** -23 * big + 2.0 ** -21
    silu = torch.full((M, N // 2), float("nan"), device=dev, dtype=torch.bfloat16)
    ops.gemm_silu(x, w, silu)
    gu = ref.view(M, N // 16, 16)
    want = (torch.nn.functional.silu(gu[..., :8]) * gu[..., 8:]).reshape(M, N // 2)
    assert float((silu - want).abs().max()) <= 2.0 ** -8 * float(want.abs().max()) + K * 2.0 ** -22 * big * big
