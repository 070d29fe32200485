"""A mixed step's attention in one launch (attention_mixed.hip) against the PyTorch reference."""
import math

import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops import reference as R

pytestmark = pytest.mark.gpu


# decode contexts on both sides of a page, an idle slot, prompts that end inside a tile, begin behind cached tokens or have one row, padded work items;
# counts of (row, kv head, partition) items that 2, 4 and 8 waves each take, and that leave groups of a workgroup without one; partitions that
# are empty; one kv head; groups of heads that go in two launches (waves 0)
@pytest.mark.parametrize("ctxs,nparts,prompts,hq,hkv,waves", [
    ([1, 31, 32, 33, 300], 1, [(45, 45)], 32, 8, 8), ([40, 700], 3, [(64, 64), (1, 90)], 32, 8, 8), ([5], 1, [(130, 200)], 4, 1, 8),
    ([17] * 49, 1, [(65, 65)], 32, 8, 4), ([33, 64] * 41, 1, [(3, 3)], 32, 8, 2), ([600] * 7, 2, [(300, 1000)], 32, 8, 8), ([77] * 3, 1, [(70, 70)], 16, 8, 0),
    ([90] * 97, 1, [(20, 20)], 4, 1, 8)])
@pytest.mark.parametrize("idle", [False, True])
def test_mixed_attention(gpu, ctxs, nparts, prompts, hq, hkv, waves, idle):
    g = torch.Generator().manual_seed(sum(ctxs) + hq + len(prompts))
    B, C = len(ctxs), sum(n for n, _ in prompts)
    lens = ctxs + [c for _, c in prompts]
    pages = [-(-n // 32) for n in lens]
    kc = torch.randn(sum(pages) + 2, hkv, 32, 128, generator=g).bfloat16()
    vc = torch.randn(sum(pages) + 2, hkv, 128, 32, generator=g).bfloat16()
    perm = torch.randperm(sum(pages) + 2, generator=g).int()
    bt = torch.zeros(len(lens) + 1, max(pages) + 1, dtype=torch.int32)
    at = 0
    for i, n in enumerate(pages):
        bt[i, :n] = perm[at:at + n]
        at += n
    q = torch.randn(B + C, hq, 128, generator=g).bfloat16()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32)  # noqa: E731
    live = torch.ones(B, dtype=torch.int32)
    if idle:
        live[B // 2] = 0
    rows = (bt[:B], torch.arange(B, dtype=torch.int32), live, i32(ctxs), torch.arange(B, dtype=torch.int32), torch.zeros(B, dtype=torch.int32))
    qs, ql, items, row = [], [], [], B
    for i, (n, _) in enumerate(prompts):
        qs.append(row)
        ql.append(n)
        items += [(i, t) for t in reversed(range(-(-n // 64)))]
        row += n
    items += [(len(prompts), 0)] * 3  # padded items point at an empty sequence
    tiles = (bt[B:], i32(qs + [0]), i32(ql + [0]), i32([c for _, c in prompts] + [0]), i32([s for s, _ in items]), i32([t for _, t in items]))
    assert torch.ops.dsse.mixed_attention_waves(B, hq, hkv, nparts, len(items)) == waves
    part = 0 if nparts > 1 else math.ceil(max(ctxs) / 128) * 128
    ref = torch.zeros_like(q)
    R.paged_attention(0, q[:B], kc, vc, *rows, ref[:B])
    R.paged_attention(2, q, kc, vc, *(t[:-1] if i in (1, 2, 3) else t[:-3] if i > 3 else t for i, t in enumerate(tiles)), ref)
    out = torch.zeros_like(q).to(gpu)
    po = torch.full((B * hkv * nparts * 16 * 128,), float("nan"), device=gpu)
    pml = torch.full((B * hkv * nparts * 32,), float("nan"), device=gpu)
    c = lambda ts: tuple(t.to(gpu).contiguous() for t in ts)  # noqa: E731
    ops.mixed_attention(q.to(gpu), kc.to(gpu), vc.to(gpu), out, po, pml, c(rows), part, nparts, c(tiles), 32 * bt.shape[1])
    keep = torch.cat([live.bool(), torch.ones(C, dtype=torch.bool)])
    # weights and values are bf16: a result's error is some 2^-8 of the largest value it averages (as in the two kernels' own tests)
    torch.testing.assert_close(out.cpu()[keep].float(), ref[keep].float(), rtol=1e-2, atol=2e-2)
    assert float(out.cpu()[~keep].float().abs().sum()) == 0
