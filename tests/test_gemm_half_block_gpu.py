"""The pipelined tiled-layout GEMM with a half-empty last column block (N % 256 == 128) in every epilogue -- fp32, added to a
residual, bf16, gated, and rotated queries and keys with the cache write -- with and without a K split, against fp64 products."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops import reference as R
from distributed_sse_for_llm_response_amd.ops.reference import tile_weight

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(1025, 128, 512), (1200, 384, 256), (600, 128, 4096), (257, 2176, 4096), (300, 8320, 2048)])
def test_half_empty_column_block(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(N + K)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    wt = tile_weight(w)
    want = x.double() @ w.double().t()
    bound = 4 * K ** 0.5 * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())  # fp32 sums of K products, in any order
    guard = torch.full((M + 1, N), 7.0, device="cuda")  # nothing may land past the last column: the next row
    out = guard[:M]
    ops.gemm_out(x, wt, out)
    assert ((out.double() - want).abs() <= bound).all() and bool((guard[M] == 7.0).all())
    ops.gemm_resid(x, wt, out)
    assert ((out.double() - 2 * want).abs() <= 2 * bound + 2.0 ** -23 * want.abs()).all()
    half = torch.zeros(M, N, device="cuda", dtype=torch.bfloat16)
    ops.gemm_out(x, wt, half)
    assert ((half.double() - want).abs() <= bound + 2.0 ** -8 * want.abs()).all()
    act = torch.zeros(M, N // 2, device="cuda", dtype=torch.bfloat16)
    ops.gemm_silu(x, wt, act)  # 16-row tiles of the weight hold 8 gate and 8 up rows
    z = want.view(M, N // 16, 2, 8)
    ref = (torch.nn.functional.silu(z[:, :, 0]) * z[:, :, 1]).reshape(M, N // 2)
    scale = (z[:, :, 0].abs() + 1) * (z[:, :, 1].abs() + 1)
    err = 2.0 ** -8 * ref.abs() + 4 * bound.amax() * scale.reshape(M, N // 2)
    assert ((act.double() - ref).abs() <= err + 1e-6).all()


# query and key/value heads of 128: 17 * 128 columns; products that the plan splits over K and one that it does not
@pytest.mark.parametrize("M,nh,nkv,K", [(300, 15, 1, 4096), (600, 1, 1, 2048), (1100, 9, 3, 512)])
def test_rotated_heads_of_a_half_empty_block(M, nh, nkv, K):
    N = (nh + 2 * nkv) * 128
    assert N % 256 == 128
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    want = x.double() @ w.double().t()
    bound = 4 * K ** 0.5 * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()).max().item()  # as above, the largest
    rope = R.rope_table(4096, 1e6, x.device)
    positions = torch.arange(M, dtype=torch.int32)
    pages = (M + 31) // 32 + 1
    slots = torch.randperm(pages * 32, generator=torch.Generator().manual_seed(K))[:M].to(torch.int32)

    def heads(device):
        return [torch.full(s, 3.0, device=device, dtype=torch.bfloat16)
                for s in ((M + 1, nh * 128), (pages, nkv, 32, 128), (pages, nkv, 128, 32))]

    got, ref = heads("cuda"), heads("cpu")
    ops.gemm_qkv_rope(x, tile_weight(w), positions.cuda(), slots.cuda(), rope, got[0][:M], got[1], got[2], nh, nkv)
    R.rope_kv_write(want.float().cpu(), positions, slots, rope.cpu(), ref[0][:M], ref[1], ref[2], nh, nkv)
    for a, b in zip(got, ref):  # a rotated element is two products' sum; two roundings to bf16 that may fall apart
        a, b = a.cpu().double(), b.double()
        assert ((a - b).abs() <= 2 * bound + 2.0 ** -7 * b.abs()).all()
