"""The shared-page form of sink attention (csrc/kernels/sink_attention.hip) with a distance bias, with one and with two column
tiles per wave, and with maxima that grow from page to page, against the op's reference."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops import layers_reference as lref

pytestmark = pytest.mark.gpu
PAGE = 32


def i32(x):
    return torch.tensor(x, dtype=torch.int32)


# few workgroups (one tile per wave) and 256 or more (two); key width = value width and not; bias tables of one entry, within
# a page, longer than the LDS strip; groups of 1, 2 and 4 heads; windows with kept first keys; scores that grow along the walk
@pytest.mark.parametrize("H,G,D,V,window,keep,rel_len,many,growth", [
    (4, 2, 128, 128, 1 << 30, 0, 118, False, 0.0), (8, 2, 64, 64, 40, 3, 1, False, 3.0), (3, 3, 96, 96, 1 << 30, 0, 0, False, 3.0),
    (4, 1, 32, 32, 33, 40, 2000, False, -2.0), (4, 2, 64, 48, 1 << 30, 0, 20, False, 3.0), (8, 8, 128, 128, 64, 5, 50, True, 3.0),
    (32, 8, 64, 64, 1 << 30, 0, 0, True, -2.0)])
def test_prompt_portions(H, G, D, V, window, keep, rel_len, many, growth):
    ql = [70, 1, 33, 16, 0] + [2, 5, 17] * 10 * many
    start = [0, 31, 64, 1100, 0] + [0, 40, 7] * 10 * many
    g = torch.Generator().manual_seed(H + D)
    n, T = len(ql), sum(ql)
    need = [-(-(a + b) // PAGE) for a, b in zip(ql, start)]
    bt, k = torch.zeros(n, max(need), dtype=torch.int32), 0
    perm = torch.randperm(sum(need) + 1, generator=g).to(torch.int32)
    for s, m in enumerate(need):
        bt[s, :m], k = perm[k:k + m], k + m
    # bf16 operands on both sides: the scores differ by fp32 rounding alone
    q = torch.randn(T, H, D, generator=g).bfloat16().float()
    kc = torch.randn(sum(need) + 1, PAGE, G, D, generator=g)
    vc = torch.randn(sum(need) + 1, PAGE, G, V, generator=g).bfloat16()
    for s, m in enumerate(need):  # score scale by page of the walk: maxima that pass the lag again and again, or never
        for j in range(m):
            kc[bt[s, j]] *= max(0.3, 1.0 + growth * j / m)
    kc = kc.bfloat16()
    vt = torch.zeros(sum(need) + 1, G, V, PAGE, dtype=torch.bfloat16)
    for off in range(PAGE):
        vt[:, :, :, lref.vt_position(off)] = vc[:, off]
    rel = torch.randn(H, rel_len, generator=g) if rel_len else None
    meta = (i32([sum(ql[:s]) for s in range(n)]), i32(ql), i32([a + b for a, b in zip(ql, start)]))
    rows = ops.sink_tile_rows(torch.bfloat16, H, G, D, V)
    items = [(s, t) for s in range(n) for t in range(-(-ql[s] // rows))]
    assert (len(items) * H * rows // 128 >= 256) == many
    sink, scale = torch.randn(H, generator=g), 1.5 * D ** -0.5
    want = torch.zeros(T, H, V, dtype=torch.float32)
    lref.sink_attention(q, kc, vc, bt, *meta, sink, None, want, window, scale, keep_first=keep, rel=rel)
    c = lambda t: None if t is None else t.cuda()  # noqa: E731
    got = torch.zeros(T, H, V, dtype=torch.bfloat16, device="cuda")
    ops.sink_attention(c(q), c(kc), c(vc), c(bt), *map(c, meta), c(i32([s for s, _ in items])), c(i32([t for _, t in items])),
                       c(sink), None, got, window, scale, rows, c(vt), keep_first=keep, rel=c(rel))
    # weights and outputs are rounded to bf16 (2^-9 each); scores below 100, so weights differ by exp(100 2^-22) besides
    assert (got.cpu().float() - want).abs().max() <= (2.0 ** -8 + 5e-5) * vc.float().abs().max()


# one and two column tiles per wave, with kept first keys and a bias
@pytest.mark.parametrize("D,V,keep,rel_len", [(128, 128, 0, 0), (64, 48, 0, 0), (64, 64, 40, 9)])
def test_pages_behind_a_window(D, V, keep, rel_len):
    """A value that is not finite reaches rows whose 32-row stretch has its page in the window, and no others: the walk of an
    item of 128 rows starts up to 127 keys ahead of a row's window."""
    T, H, window, bad = 400, 2, 64, 80
    g = torch.Generator().manual_seed(D + V)
    pages = -(-T // PAGE)
    kc = torch.randn(pages, PAGE, H, D, generator=g).bfloat16().cuda()
    vt = torch.randn(pages, H, V, PAGE, generator=g).bfloat16().cuda()
    bt = torch.arange(pages, dtype=torch.int32)[None].cuda()
    q, sink = torch.randn(T, H, D, generator=g).cuda(), torch.randn(H, generator=g).cuda()
    rel = torch.randn(H, rel_len, generator=g).cuda() if rel_len else None
    rows = ops.sink_tile_rows(torch.bfloat16, H, H, D, V)
    assert rows == 128
    items = list(range(-(-T // rows)))
    meta = [t.cuda() for t in (i32([0]), i32([T]), i32([T]), i32([0] * len(items)), i32(items))]
    outs = []
    for x in (0.0, float("nan")):
        vt[bad // PAGE, :, :, lref.vt_position(bad % PAGE)] = x
        out = torch.zeros(T, H, V, dtype=torch.bfloat16, device="cuda")
        # the kernel reads values from the transposed pages alone
        ops.sink_attention(q, kc, torch.zeros(pages, PAGE, H, V, dtype=torch.bfloat16, device="cuda"), bt, *meta, sink, None, out,
                           window, D ** -0.5, rows, vt, keep_first=keep, rel=rel)
        outs.append(out.cpu())
    clean, got = outs
    far = torch.ones(T, dtype=torch.bool)
    far[bad // PAGE * PAGE:(bad // PAGE + 1) * PAGE + window] = False   # rows 64 .. 159
    assert torch.isfinite(clean).all() and torch.equal(got[far], clean[far])
    assert torch.isnan(got[bad:bad + window].float()).all()
