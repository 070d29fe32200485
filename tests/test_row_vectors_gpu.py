"""Row-wise kernels in groups of four elements, rows over several workgroups or in registers, against their references at the
edges of the split: single groups, widths that are no multiple of four (the scalar forms), the widest rows in registers and one
group more, few rows and many."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops import layers_reference as lref

pytestmark = pytest.mark.gpu
EPS = 1e-5


def c(t):
    return None if t is None else t.cuda()


def near(got, want, steps):
    """Within `steps` roundings of the result's type of the largest value."""
    unit = 2.0 ** -9 if got.dtype == torch.bfloat16 else 2.0 ** -24
    assert (got.cpu().double() - want.double()).abs().max() <= steps * unit * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("M,W", [(1, 4), (3, 6), (2, 1020), (16, 4096), (513, 1028), (2, 16384), (2, 16388)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_stream_rows(M, W, dtype):
    g = torch.Generator().manual_seed(W)
    rn = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    resid, y, y3, w, b, vec, alpha = rn(M, W), rn(M, W), rn(3 * M, W), rn(W), rn(W), rn(W), torch.tensor([0.7])
    embed, ids, gain = rn(5, W).to(dtype), torch.randint(0, 5, (M,), generator=g, dtype=torch.int32), torch.tensor([1.3]).to(dtype)
    # a few fp32 operations per element on values below 20; tanhf is good to two units of the last place
    for args in ((y, 0.5, embed, vec, True), (None, 1.0, None, None, True), (y, 2.0, None, None, False)):
        r0, r1, x0, x1 = resid.clone(), c(resid), torch.zeros(M, W, dtype=dtype), torch.zeros(M, W, dtype=dtype, device="cuda")
        norm = (alpha, w, b) if args[4] else (None, None, None)
        lref.stream_step(args[0], args[1], r0, ids, args[2], args[3], *norm, x0 if args[4] else None)
        ops.stream_step(c(args[0]), args[1], r1, c(ids), c(args[2]), c(args[3]), *map(c, norm), x1 if args[4] else None)
        near(r1, r0, 4)
        near(x1, x0, 2 if dtype == torch.bfloat16 else 40)
    # a sum of W squares: at most W / 256 + 16 roundings in a row, halved by the square root
    steps = W / 256 + 24
    for src, n in ((y, 1), (y3, 3), (None, 1)):
        r0, r1, x0, x1 = resid.clone(), c(resid), torch.zeros(M, W, dtype=dtype), torch.zeros(M, W, dtype=dtype, device="cuda")
        lref.scalar_norm(src, gain, r0, x0, EPS, n)
        ops.scalar_norm(c(src), c(gain), r1, x1, EPS, n)
        near(r1, r0, steps)
        near(x1, x0, 2 if dtype == torch.bfloat16 else steps)
    e0, e1 = torch.zeros(M, W), torch.zeros(M, W, device="cuda")
    lref.embed_rows(ids, embed, e0, None, 0.3)
    ops.embed_rows(c(ids), c(embed), e1, None, 0.3)
    near(e1, e0, 2)
    if dtype == torch.float32:
        want = torch.zeros(M, W)
        lref.rms_mix(y, w, resid, b, EPS, 0.5, want)
        out = c(y)
        ops.rms_mix(out, c(w), c(resid), c(b), EPS, 0.5, out)  # in place
        near(out, want, 2 * steps)


@pytest.mark.parametrize("T,nh,D", [(1, 1, 6), (5, 3, 64), (2, 16, 128), (3, 37, 32), (513, 5, 128), (700, 37, 32), (1500, 19, 6), (3001, 41, 6)])
@pytest.mark.parametrize("kind", [0, 1, 2, 3])
def test_heads_over_workgroups_and_waves(T, nh, D, kind):
    g = torch.Generator().manual_seed(nh + D)
    x = torch.randn(T, nh, D, generator=g)
    w = torch.randn(nh * D if kind == 1 else D, generator=g) if kind in (1, 3) else None
    rope, pos = torch.randn(9, D // 2 - 1, 2, generator=g), torch.randint(0, 9, (T,), generator=g, dtype=torch.int32)
    rows = torch.randperm(T, generator=g).to(torch.int32)
    rows[0] = -1
    want, got = torch.zeros(T, nh, D), torch.zeros(T, nh, D, device="cuda")
    lref.norm_rope_rows(x, w, pos, rope, want, rows, kind, EPS, 0.4)
    ops.norm_rope_rows(c(x), c(w), c(pos), c(rope), got, c(rows), kind, EPS, 0.4)
    near(got, want, nh * D / 256 + 24)


@pytest.mark.parametrize("C,K,off", [(8, 4, 4), (1028, 4, 0), (12, 4, 3), (8, 3, 0)])
@pytest.mark.parametrize("act", [0, 1, 2])
def test_convolution_rows(C, K, off, act):
    """Portions around the eight rows of a workgroup, shorter than the taps, continued and fresh; a misaligned column slice and
    three taps take the scalar form."""
    g = torch.Generator().manual_seed(C)
    ql, ctx, slot = [9, 1, 16, 0, 2], [9, 5, 40, 3, 2], [1, 0, 4, 3, 2]
    T, qs = sum(ql), [0, 9, 10, 26, 26]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32)  # noqa: E731
    meta = (i32(qs), i32(ql), i32(ctx), i32(slot))
    wide = torch.randn(T, C + 8, generator=g)
    taps, bias, ib = (torch.randn(*s, generator=g) for s in ((C, K), (C,), (C,)))
    tail = torch.randn(5, K - 1, C, generator=g)
    t0, t1, o0, o1 = tail.clone(), c(tail), torch.zeros(T, C), torch.zeros(T, C, device="cuda")
    lref.conv_state(wide[:, off:off + C], taps, bias, t0, *meta, o0, None, ib, act)
    ops.conv_state(c(wide)[:, off:off + C], c(taps), c(bias), t1, *map(c, meta), o1, None, c(ib), act)
    near(o1, o0, 30)  # six products and sums, an exponential
    near(t1, t0, 2)


@pytest.mark.parametrize("T", [255, 256, 259])
def test_recurrence_coefficients_of_several_rows(T):
    g = torch.Generator().manual_seed(T)
    blocks, bw = 3, 100
    C = blocks * bw
    i32 = lambda v: torch.tensor(v, dtype=torch.int32)  # noqa: E731
    meta = (i32([0]), i32([T]), i32([T]), i32([0]))
    u, y, lam = torch.randn(T, C, generator=g), torch.randn(T, C, generator=g), torch.randn(C, generator=g)
    gates = torch.randn(T, blocks, 2 * bw, generator=g)
    s0, s1, o0, o1 = torch.zeros(1, C), torch.zeros(1, C, device="cuda"), torch.zeros(T, C), torch.zeros(T, C, device="cuda")
    lref.lru_scan(u, gates.clone(), y, lam, s0, *meta, o0, 8.0)
    ops.lru_scan(c(u), c(gates), c(y), c(lam), s1, *map(c, meta), o1, 8.0)
    near(o1, o0, 400)  # decays below one: errors of some ten operations per step, damped, over the steps they last
    near(s1, s0, 400)
