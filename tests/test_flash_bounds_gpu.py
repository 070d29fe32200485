"""Flash prefill: what a token holds does not reach queries in whose key blocks it is not, also where it is not a finite number."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops import reference as R

pytestmark = pytest.mark.gpu


# 64 queries behind `before` cached tokens: the last block of 64 keys begins after the first 32 of them (32), or inside them (0, 63); a split of the keys whose
# second part only the last 32 see
@pytest.mark.parametrize("before,n,hq,hkv", [(32, 64, 32, 8), (32, 64, 16, 8), (32, 64, 8, 8), (96, 40, 4, 1), (0, 64, 32, 8), (63, 64, 32, 8), (288, 200, 32, 8)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("split", [False, True])
def test_values_after_a_query(gpu, before, n, hq, hkv, bad, split):
    g = torch.Generator().manual_seed(before + n)
    ctx = before + n
    pages = -(-ctx // 32)
    kc = torch.randn(pages, hkv, 32, 128, generator=g).bfloat16()
    vc = torch.randn(pages, hkv, 128, 32, generator=g).bfloat16()
    q = torch.randn(n, hq, 128, generator=g).bfloat16()
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32)  # noqa: E731
    tiles = list(range(-(-n // 64)))
    meta = (torch.arange(pages, dtype=torch.int32)[None], i32(0), i32(n), i32(ctx))
    work = (i32(*[0] * len(tiles)), i32(*tiles))
    ref = torch.zeros_like(q)
    R.paged_attention(2, q, kc, vc, *meta, *work, ref, None, None, 32 * pages, 1)
    last = (ctx - 1) // 64  # the last block of 64 keys
    vc[2 * last:] = bad
    out = torch.zeros_like(q).to(gpu)
    c = lambda ts: tuple(t.to(gpu) for t in ts)  # noqa: E731
    if not split:
        ops.paged_attention(2, q.to(gpu), kc.to(gpu), vc.to(gpu), *c(meta), *c(work), out, torch.zeros(1, device=gpu), torch.zeros(1, device=gpu), 32 * pages, 1)
    else:  # every tile's keys up to the last block, and the rest, which for the first tiles is empty
        nt = len(tiles)
        seq, tile = [0] * (2 * nt), [t for t in tiles for _ in range(2)]
        kb = [v for _ in tiles for v in (0, last, last, last + 1)]
        w = i32(*seq, *tile, *kb, *range(2 * nt)).to(gpu)
        comb = i32(*[v for t in tiles for v in (0, t, 2 * t, 2)]).to(gpu)
        po = torch.full((2 * nt * hq * 64 * 128,), float("nan"), device=gpu)
        pml = torch.full((2 * nt * hq * 64 * 2,), float("nan"), device=gpu)
        ops.flash_prefill_split(q.to(gpu), kc.to(gpu), vc.to(gpu), *c(meta), w, comb, out, po, pml, 2 * nt)
    # queries go in groups of 32: those whose last position is before the block
    clean = [i for i in range(n) if before + min(n, i // 32 * 32 + 32) - 1 < 64 * last]
    torch.testing.assert_close(out.cpu()[clean].float(), ref[clean].float(), rtol=1e-2, atol=2e-2)
    seen = [i for i in range(n) if before + i >= 64 * last]
    assert not torch.isfinite(out.cpu()[seen].float()).any()
