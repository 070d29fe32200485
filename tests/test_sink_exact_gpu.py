"""Sink attention of prompt portions in the exact mode on the fp32 matrix cores (csrc/kernels/sink_exact.hip) against the op's
reference, with every option of the row kernel that it takes."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops import layers_reference as lref

pytestmark = pytest.mark.gpu
PAGE = 32


def i32(x):
    return torch.tensor(x, dtype=torch.int32)


# groups of 4, 2 and 1 heads; key width = value width and not; windows with kept keys; bias tables of one entry and long; caps;
# a gate per head and per element; output rows that are a slice of wider ones
@pytest.mark.parametrize("H,G,D,V,window,keep,rel_len,cap,gates", [
    (4, 1, 128, 128, 1 << 30, 0, 0, 0.0, 0), (4, 2, 64, 64, 33, 40, 1, 0.0, 1), (3, 3, 16, 16, 1, 2, 0, 5.0, 2),
    (8, 2, 32, 112, 64, 0, 300, 0.0, 2), (2, 1, 96, 96, 1 << 30, 0, 7, 20.0, 1)])
def test_prompt_portions(H, G, D, V, window, keep, rel_len, cap, gates):
    ql, start = [70, 1, 33, 16, 0, 5], [0, 31, 64, 500, 0, 3]
    g = torch.Generator().manual_seed(H + D)
    n, T = len(ql), sum(ql)
    need = [-(-(a + b) // PAGE) for a, b in zip(ql, start)]
    bt, k = torch.zeros(n, max(need), dtype=torch.int32), 0
    perm = torch.randperm(sum(need) + 1, generator=g).to(torch.int32)
    for s, m in enumerate(need):
        bt[s, :m], k = perm[k:k + m], k + m
    q = torch.randn(T, H, D, generator=g)
    kc, vc = (torch.randn(sum(need) + 1, PAGE, G, w, generator=g) for w in (D, V))
    rel = torch.randn(H, rel_len, generator=g) if rel_len else None
    sink = torch.randn(H, generator=g) if gates != 1 else None
    gate = torch.randn(T, (0, H, H * V)[gates] + 3, generator=g)[:, 3:] if gates else None
    meta = (i32([sum(ql[:s]) for s in range(n)]), i32(ql), i32([a + b for a, b in zip(ql, start)]))
    rows = ops.sink_tile_rows(torch.float32, H, G, D, V)
    assert rows == {1: 64, 2: 32, 4: 16}[H // G]
    items = [(s, t) for s in range(n) for t in range(-(-ql[s] // rows))]
    scale = D ** -0.5
    want = torch.zeros(T, H, V)
    lref.sink_attention(q, kc, vc, bt, *meta, sink, gate, want, window, scale, softcap=cap, keep_first=keep, rel=rel, out_scale=0.7)
    c = lambda t: None if t is None else t.cuda()  # noqa: E731
    wide = torch.full((T, H * V + 5), 9.0, device="cuda")
    got = wide[:, 2:2 + H * V].unflatten(1, (H, V))
    ops.sink_attention(c(q), c(kc), c(vc), c(bt), *map(c, meta), c(i32([s for s, _ in items])), c(i32([t for _, t in items])),
                       c(sink), c(gate), got, window, scale, rows, softcap=cap, keep_first=keep, rel=c(rel), out_scale=0.7)
    # scores: sums of D products, D 2^-24 of |q||k| scale < 10 each, times a factor e^s; outputs: 600 weights.  Both sides round.
    assert (got.cpu() - want).abs().max() <= 2 * (10 * D + 600) * 2.0 ** -24 * vc.abs().max()
    assert (wide[:, :2] == 9.0).all() and (wide[:, 2 + H * V:] == 9.0).all()


@pytest.mark.parametrize("H,G,D,V,window,keep", [(4, 2, 64, 64, 1 << 30, 0), (4, 1, 128, 96, 40, 3), (2, 2, 16, 128, 20, 0)])
@pytest.mark.parametrize("bad", ["nan", "inf"])
def test_values_that_a_row_does_not_see(H, G, D, V, window, keep, bad):
    """Values that are not finite where a row sees nothing -- later tokens, keys behind the window, places past the context that
    an earlier owner of the page left -- do not reach it; where it sees them they do."""
    ql, start = [50, 9, 33], [0, 31, 100]
    g = torch.Generator().manual_seed(D + V)
    n, T = len(ql), sum(ql)
    need = [-(-(a + b) // PAGE) for a, b in zip(ql, start)]
    bt, k = torch.zeros(n, max(need), dtype=torch.int32), 0
    for s, m in enumerate(need):
        bt[s, :m], k = torch.arange(k, k + m, dtype=torch.int32), k + m
    q = torch.randn(T, H, D, generator=g)
    kc, vc = (torch.randn(sum(need), PAGE, G, w, generator=g) for w in (D, V))

    def place(s, j):
        return int(bt[s, j // PAGE]), j % PAGE

    vc[place(0, 20) + (0, 5)] = float(bad)       # rows 20 .. of the first sequence see it, until the window has passed
    vc[place(2, 10) + (G - 1, V - 1)] = float(bad)  # behind the window of some cases
    for s in range(n):                            # the rest of the last pages
        for j in range(ql[s] + start[s], need[s] * PAGE):
            kc[place(s, j)] = vc[place(s, j)] = float(bad)
    meta = (i32([sum(ql[:s]) for s in range(n)]), i32(ql), i32([a + b for a, b in zip(ql, start)]))
    rows = ops.sink_tile_rows(torch.float32, H, G, D, V)
    items = [(s, t) for s in range(n) for t in range(-(-ql[s] // rows))]
    sink, gate = torch.randn(H, generator=g), torch.randn(T, H, generator=g)
    want = torch.zeros(T, H, V)
    lref.sink_attention(q, kc, vc, bt, *meta, sink, gate, want, window, D ** -0.5, keep_first=keep)
    c = lambda t: t.cuda()  # noqa: E731
    got = torch.zeros(T, H, V, device="cuda")
    ops.sink_attention(c(q), c(kc), c(vc), c(bt), *map(c, meta), c(i32([s for s, _ in items])), c(i32([t for _, t in items])),
                       c(sink), c(gate), got, window, D ** -0.5, rows, keep_first=keep)
    fine = torch.isfinite(want)
    assert fine.any() and not fine.all() and torch.equal(torch.isfinite(got.cpu()), fine)
    assert (got.cpu() - want)[fine].abs().max() <= 2 * (10 * D + 600) * 2.0 ** -24 * 5   # as above; |v| < 5


@pytest.mark.parametrize("H,G,D,V,window,keep,rel_len", [(4, 2, 128, 128, 1 << 30, 0, 0), (4, 1, 64, 64, 70, 40, 9), (2, 2, 32, 48, 200, 0, 0)])
def test_rows_do_not_depend_on_the_cut(H, G, D, V, window, keep, rel_len):
    """The same rows bit for bit, whatever portions their prompt comes in: sums are grouped by pages of the sequence."""
    T = 420
    g = torch.Generator().manual_seed(D)
    pages = -(-T // PAGE)
    bt = torch.randperm(pages, generator=g).to(torch.int32)[None].cuda()
    q = torch.randn(T, H, D, generator=g).cuda()
    kc, vc = (torch.randn(pages, PAGE, G, w, generator=g).cuda() for w in (D, V))
    sink = torch.randn(H, generator=g).cuda()
    rel = torch.randn(H, rel_len, generator=g).cuda() if rel_len else None
    rows = ops.sink_tile_rows(torch.float32, H, G, D, V)
    outs = []
    for cut in ([T], [1, 37, 130, 2, 64, 186], [33] * 12 + [24]):
        out, at = torch.zeros(T, H, V, device="cuda"), 0
        for n in cut:
            items = range(-(-n // rows))
            meta = (i32([0]), i32([n]), i32([at + n]), i32([0] * len(items)), i32(list(items)))
            ops.sink_attention(q[at:at + n], kc, vc, bt, *(t.cuda() for t in meta), sink, None, out[at:at + n], window,
                               D ** -0.5, rows, keep_first=keep, rel=rel)
            at += n
        outs.append(out)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
