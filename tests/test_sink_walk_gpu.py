"""The decode form of the sink attention reads its pages in two ways (allocating in the caches, or past them) chosen by the bytes
of a launch's walks, and counts the keys' steps at compile time when keys and values are of one width; decode_prep leaves the
tokens of all live sequences behind."""
import math

import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops import layers_reference as lref

PAGE = 32


def i32(x):
    return torch.tensor(x, dtype=torch.int32)


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D,V,window,nparts", [(16, 8, 128, 128, 10 ** 9, 1), (16, 8, 128, 128, 10 ** 9, 3), (8, 2, 64, 64, 45, 1),
                                                   (34, 1, 32, 32, 10 ** 9, 1), (4, 2, 64, 128, 10 ** 9, 1), (8, 2, 256, 256, 10 ** 9, 1),
                                                   (4, 4, 96, 96, 33, 2)])
def test_both_walks(H, G, D, V, window, nparts):
    """One key, one page, a page and a key, more pages than the eight waves, an idle row between them: past the caches bit for
    bit what allocating loads give, both near the reference (weights in bf16: 2^-9 of an output, plus the output's rounding)."""
    g = torch.Generator().manual_seed(5)
    ctx, ql = [1, 32, 33, 0, 700, 290], [1, 1, 1, 0, 1, 1]
    need = [math.ceil(n / PAGE) for n in ctx]
    perm, bt, k = torch.randperm(sum(need), generator=g).tolist(), torch.zeros(6, max(need), dtype=torch.int32), 0
    for s, n in enumerate(need):
        bt[s, :n], k = i32(perm[k:k + n]), k + n
    q = torch.randn(6, H, D, generator=g)
    kc, vc = (torch.randn(sum(need), PAGE, G, n, generator=g).to(torch.bfloat16) for n in (D, V))
    vt = torch.zeros(sum(need), G, V, PAGE, dtype=torch.bfloat16)
    for off in range(PAGE):
        vt[:, :, :, lref.vt_position(off)] = vc[:, off]
    sink, gate, scale = torch.randn(H, generator=g), torch.randn(6, H, generator=g), D ** -0.5
    meta = (i32([0, 1, 2, 3, 4, 5]), i32(ql), i32(ctx))
    want = torch.zeros(6, H, V, dtype=torch.bfloat16)
    lref.sink_attention(q, kc, vc, bt, *meta, sink, gate, want, window, scale, vt)
    c = lambda t: t.cuda()  # noqa: E731
    args = [c(t) for t in (q, kc, vc, bt, *meta, i32(range(6)), i32([0] * 6), sink, gate)]
    tokens = sum(min(n, window) for n in ctx)
    bytes_ = tokens * G * (D + V) * 2
    got = []
    for walked, once in ((None, 0.0), (i32([sum(ctx)]).cuda(), 0.9 * bytes_), (i32([sum(ctx)]).cuda(), 6.0 * bytes_)):
        out = torch.zeros(6, H, V, dtype=torch.bfloat16, device="cuda")
        part = torch.zeros(6 * H * nparts * (V + 2), device="cuda") if nparts > 1 else None
        ops.sink_attention(*args, out, window, scale, 1, c(vt), part=part, nparts=nparts, walked=walked, once=once)
        got.append(out.cpu())
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])
    live = [i for i, n in enumerate(ql) if n]
    torch.testing.assert_close(got[0][live].float(), want[live].float(), atol=2e-2, rtol=2e-2)


def _prep(B, dev):
    g = torch.Generator().manual_seed(B)
    active = (torch.rand(B, generator=g) < 0.7).to(torch.int32)
    pos = torch.randint(0, 4 * PAGE, (B,), generator=g, dtype=torch.int32)
    bt = torch.randint(0, 50, (B, 4), generator=g, dtype=torch.int32)
    outs = [torch.zeros(B, dtype=torch.int32, device=dev) for _ in range(3)]
    walked = torch.full((1,), -7, dtype=torch.int32, device=dev)
    ops.decode_prep(active.to(dev), pos.to(dev), bt.to(dev), *outs, 50, walked)
    assert int(walked) == int(((pos + 1) * active).sum())
    live = active.bool()
    page = bt.gather(1, (pos // PAGE).long()[:, None])[:, 0]
    slots, ctx, ql = (o.cpu() for o in outs)
    assert torch.equal(slots, torch.where(live, page * PAGE + pos % PAGE, torch.full_like(pos, -1)))
    assert torch.equal(ctx, torch.where(live, pos + 1, torch.zeros_like(pos))) and torch.equal(ql, active)


@pytest.mark.parametrize("B", [1, 65])
def test_tokens_of_a_step(B):
    _prep(B, "cpu")


@pytest.mark.gpu
@pytest.mark.parametrize("B", [1, 64, 65, 1024, 1500])
def test_tokens_of_a_step_gpu(B):
    _prep(B, "cuda")
