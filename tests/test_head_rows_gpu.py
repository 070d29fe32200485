"""Heads in pieces of four numbers: norms and rotations with a head's lanes side by side, values written page by page, gated head
norms -- at the narrowest and widest heads of that form, more heads than a walk takes, partial rotations, rows that make whole pages
and rows that do not."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops import layers_reference as lref

pytestmark = pytest.mark.gpu
EPS = 1e-5
PAGE = 32


def c(t):
    return None if t is None else t.cuda()


def near(got, want, steps):
    """Within `steps` roundings of the result's type of the largest value."""
    unit = 2.0 ** -9 if got.dtype == torch.bfloat16 else 2.0 ** -24
    assert (got.cpu().double() - want.double()).abs().max() <= steps * unit * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("T,nh,D,half", [(1, 1, 32, 4), (3, 9, 32, 16), (65, 16, 128, 64), (64, 5, 64, 8), (700, 3, 256, 128), (130, 33, 64, 0)])
@pytest.mark.parametrize("kind", [0, 1, 2, 3])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_heads_in_fours(T, nh, D, half, kind, dtype):
    g = torch.Generator().manual_seed(T + D)
    wide = torch.randn(T, nh * D + 8, generator=g)
    w = torch.randn(nh * D if kind == 1 else D, generator=g) if kind in (1, 3) else None
    rope = torch.randn(11, half, 2, generator=g) if half else None
    pos = torch.randint(-1, 13, (T,), generator=g, dtype=torch.int32)  # clamped into the table
    steps = nh * D / 256 + 24  # a row's squares in sequence, the root, a rotation
    want, got = torch.zeros(T, nh, D, dtype=dtype), torch.zeros(T, nh, D, dtype=dtype, device="cuda")
    view = lambda t: t[:, 4:4 + nh * D].unflatten(1, (nh, D))  # noqa: E731
    lref.norm_rope_rows(view(wide), w, pos, rope, want, None, kind, EPS, 0.7)
    dev = c(wide)
    ops.norm_rope_rows(view(dev), c(w), c(pos), c(rope), got, None, kind, EPS, 0.7)
    near(got, want, 2 if dtype == torch.bfloat16 else steps)
    if dtype == torch.float32:  # in place: nothing beside the heads changes
        ops.norm_rope_rows(view(dev), c(w), c(pos), c(rope), view(dev), None, kind, EPS, 0.7)
        near(view(dev), want, steps)
        assert torch.equal(dev[:, :4].cpu(), wide[:, :4]) and torch.equal(dev[:, -4:].cpu(), wide[:, -4:])


@pytest.mark.parametrize("nh,D", [(1, 32), (3, 64), (8, 128), (2, 256)])
@pytest.mark.parametrize("T", [127, 128, 200])
def test_values_page_by_page(nh, D, T):
    """Rows 0-31 a whole page, 32-63 the same shifted by a token, then one page backwards, skipped and out-of-range rows, a rest."""
    g = torch.Generator().manual_seed(nh * D + T)
    rows = torch.full((T,), -1, dtype=torch.int32)
    rows[:32] = torch.arange(32) + 2 * PAGE
    rows[32:63] = torch.arange(31) + 3 * PAGE + 1
    rows[63] = 4 * PAGE + 5
    rows[64:96] = torch.arange(31, -1, -1) + 5 * PAGE
    rows[100:T] = torch.arange(T - 100) + 6 * PAGE + (7 if T < 128 else 0)
    x = torch.randn(T, nh, D, generator=g)
    pos = torch.zeros(T, dtype=torch.int32)
    pages = int(rows.max()) // PAGE + 2
    out, out_t = torch.full((pages, PAGE, nh, D), 7.0).to(torch.bfloat16), torch.full((pages, nh, D, PAGE), 7.0).to(torch.bfloat16)
    rows[97] = pages * PAGE + 3
    assert rows[rows >= 0].unique().numel() == int((rows >= 0).sum())
    got, got_t = c(out.clone()), c(out_t.clone())
    lref.norm_rope_rows(x, None, pos, None, out, rows, 0, 0.0, 1.0, out_t)
    ops.norm_rope_rows(c(x), None, c(pos), None, got, c(rows), 0, 0.0, 1.0, got_t)
    assert torch.equal(got.cpu(), out) and torch.equal(got_t.cpu(), out_t)


@pytest.mark.parametrize("M,H,V", [(1, 1, 32), (5, 3, 64), (33, 7, 128), (2, 5, 256)])
@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gated_heads_in_fours(M, H, V, kind, dtype):
    g = torch.Generator().manual_seed(M + V)
    o, wide = torch.randn(M, H, V, generator=g), torch.randn(M, H * V + 8, generator=g)
    for w in (torch.randn(V, generator=g), None):
        want, got = torch.zeros(M, H * V, dtype=dtype), torch.zeros(M, H * V, dtype=dtype, device="cuda")
        lref.gated_head_norm(o, w, wide[:, 4:4 + H * V], EPS, want, kind)
        ops.gated_head_norm(c(o), c(w), c(wide)[:, 4:4 + H * V], EPS, got, kind)
        near(got, want, 2 if dtype == torch.bfloat16 else 30)  # 32-256 squares, a root, an exponential, four products


@pytest.mark.parametrize("H,G,D,V", [(1, 1, 4, 0), (3, 2, 8, 4), (2, 1, 128, 0), (5, 1, 132, 64)])
@pytest.mark.parametrize("K", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_convolved_rows_in_fours(H, G, D, V, K, dtype):
    """Prompt portions that start, continue, are shorter than the taps, one inactive; a skipped row and one out of the pages."""
    i32 = lambda v: torch.tensor(v, dtype=torch.int32)  # noqa: E731
    g = torch.Generator().manual_seed(D + K)
    C, VW, lens, ctx = (H + G) * D, V or D, [9, 2, 0, 41], [9, 35, 3, 73]
    T, qs = sum(lens), [0, 9, 11, 11]
    x = torch.randn(T, 4 + C + G * V + 4, generator=g)
    taps = torch.randn(C, K, generator=g) if K else None
    tail = torch.randn(5, K - 1, C, generator=g) if K > 1 else None
    rope = torch.randn(70, 2 if D < 128 else 64, 2, generator=g)  # shorter than the last position
    factor = torch.rand(60, generator=g) if V else None
    slots = torch.cat([96 * s + torch.arange(n - m, n, dtype=torch.int32) for s, (m, n) in enumerate(zip(lens, ctx))]).to(torch.int32)
    slots[-1], slots[3] = 96 * 4 + 7, -1
    caches = [torch.zeros(12, PAGE, G, D, dtype=dtype), torch.zeros(12, PAGE, G, VW, dtype=dtype), torch.zeros(12, G, VW, PAGE, dtype=dtype)]
    for qt in (4, 16):
        want, got = [t.clone() for t in caches], [c(t) for t in caches]
        q_ref, q, t0, t1 = torch.zeros(T, H, D), torch.zeros(T, H, D, device="cuda"), None if tail is None else tail.clone(), c(tail)
        meta = (i32(qs), i32(lens), i32(ctx), i32([4, 0, 2, 1]))
        work = [(s, t) for s, n in enumerate(lens) for t in range(-(-n // qt))]
        lref.conv_qkv_rows(x[:, 4:], taps, t0, *meta, H, G, D, V, rope, factor, slots, q_ref, *want)
        ops.conv_qkv_rows(c(x)[:, 4:], c(taps), t1, *map(c, meta), c(i32([s for s, _ in work])), c(i32([t for _, t in work])), qt, H, G,
                          D, V, c(rope), c(factor), c(slots), q, *got)
        near(q, q_ref, 12)  # four products and sums, a rotation, a factor
        for a, r in zip(got, want):
            near(a, r, 12 if dtype == torch.float32 else 2)
        if K > 1:
            assert torch.equal(t1.cpu(), t0)


@pytest.mark.parametrize("D,half", [(32, 4), (64, 8), (128, 32)])
@pytest.mark.parametrize("kind", [0, 1, 3])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_what_is_not_finite_stays_where_it_was(D, half, kind, bad):
    """A partial rotation beside an infinite or undefined number: of the numbers that are not rotated only that one is touched (no
    norm), or what the reference says (a norm carries it through its sum)."""
    g = torch.Generator().manual_seed(D)
    x = torch.randn(5, 3, D, generator=g)
    x[1, 1, 2 * half] = bad          # the first number past the rotated ones
    x[2, 0, D - 1] = bad
    x[3, 2, 1] = bad                 # a rotated one: its partner too
    w = torch.randn(3 * D if kind == 1 else D, generator=g) if kind else None
    rope, pos = torch.randn(7, half, 2, generator=g), torch.arange(5, dtype=torch.int32)
    want, got = torch.zeros(5, 3, D), torch.zeros(5, 3, D, device="cuda")
    lref.norm_rope_rows(x, w, pos, rope, want, None, kind, EPS, 0.7)
    ops.norm_rope_rows(c(x), c(w), c(pos), c(rope), got, None, kind, EPS, 0.7)
    got = got.cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    ok = torch.isfinite(want)
    near(got[ok], want[ok], 24)


@pytest.mark.parametrize("nh,D", [(1, 32), (3, 32), (3, 64), (8, 128), (5, 256), (40, 64)])
def test_pages_that_begin_anywhere_in_the_launch(nh, D):
    """Decode rows in pages of their own, then prompts of whole and partial pages that begin at no multiple of 32 packed rows, a page
    whose first rows are not in the launch, and one whose last are not."""
    g = torch.Generator().manual_seed(nh + D)
    rows = [PAGE * (20 + b) + (5 * b) % PAGE for b in range(7)] + list(range(PAGE * 40 + 9, PAGE * 42))  # the rest of a page, then a whole one
    rows += list(range(71)) + [PAGE * 60 + 1, PAGE * 60] + list(range(PAGE * 10, PAGE * 10 + 64)) + list(range(PAGE * 50, PAGE * 50 + 30))
    T, pages = len(rows), 62
    assert T >= 128 and len(set(rows)) == T
    rows = torch.tensor(rows, dtype=torch.int32)
    x, pos = torch.randn(T, nh * D + 4, generator=g)[:, 4:].unflatten(1, (nh, D)), torch.zeros(T, dtype=torch.int32)
    out, out_t = torch.full((pages, PAGE, nh, D), 7.0).to(torch.bfloat16), torch.full((pages, nh, D, PAGE), 7.0).to(torch.bfloat16)
    got, got_t = c(out.clone()), c(out_t.clone())
    lref.norm_rope_rows(x, None, pos, None, out, rows, 0, 0.0, 0.5, out_t)
    wide = torch.zeros(T, nh * D + 4, device="cuda")
    wide[:, 4:] = c(x.flatten(1))
    ops.norm_rope_rows(wide[:, 4:].unflatten(1, (nh, D)), None, c(pos), None, got, c(rows), 0, 0.0, 0.5, got_t)
    assert torch.equal(got.cpu(), out) and torch.equal(got_t.cpu(), out_t)
