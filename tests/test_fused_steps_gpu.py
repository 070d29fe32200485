"""Launches that were joined: the linear recurrence with its coefficients, expert choice with the work list."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops import layers_reference as lref

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    ops.load_library(required=True)


def one_launch(rows, n, longest):
    """Whether a step takes coefficients and walk in one launch (csrc/kernels/recurrent.hip): by its longest sequence."""
    return (longest or rows) <= (max(24, min(48, n // 4)) if rows >= 128 else 8)


def c(t):
    return None if t is None else t.cuda()


def i32(v):
    return torch.tensor(v, dtype=torch.int32)


# one row and none per sequence; the longest one on both sides of the one-launch form, alone and beside many of one row, below and
# from the rows of the chunks; chunks of 32 rows around their edges, folded (up to 32 chunks) and carried; sequences that go on and
# ones that start; channels beyond a workgroup's 256
@pytest.mark.parametrize("ql,ctx", [
    ([1, 1, 0, 1], [7, 1, 3, 900]), ([4, 1, 8, 3], [4, 90, 8, 70]), ([5], [9]), ([9], [9]), ([96, 33], [96, 60]), ([1, 31, 32, 65], [5, 31, 40, 65]),
    ([1] * 40 + [8], [9] * 40 + [8]), ([1] * 40 + [9], [9] * 40 + [30]), ([1] * 63 + [190], [9] * 63 + [190]), ([24] * 7, [24] * 3 + [50] * 4),
    ([1] * 110 + [24], [9] * 110 + [24]), ([1] * 110 + [28], [9] * 110 + [28]), ([1] * 128 + [32], [9] * 128 + [40]),
    ([1024], [1024]), ([1000, 25], [1005, 25]), ([1, 1100], [8, 1100])])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_recurrence_that_holds_all_rows(ql, ctx, dtype):
    g = torch.Generator().manual_seed(sum(ql))
    blocks, bw = 3, 100
    C, T, n = blocks * bw, sum(ql), len(ql)
    meta = (i32([sum(ql[:i]) for i in range(n)]), i32(ql), i32(ctx), i32(list(range(n))[::-1]))
    u, y, state = torch.randn(T, C, generator=g), torch.randn(T, C, generator=g), torch.randn(n, C, generator=g)
    lam, yb = (torch.randn(C, generator=g).to(dtype) for _ in range(2))
    gates = torch.randn(T, blocks, 2 * bw, generator=g)
    s0, o0 = state.clone(), torch.zeros(T, C, dtype=dtype)
    lref.lru_scan(u, gates.clone(), y, lam, s0, *meta, o0, 8.0, yb)
    outs = []
    for alone, longest in ((False, 0), (True, 0), (True, max(ql))):
        s1, o1, made = c(state), torch.full((T, C), float("nan"), dtype=dtype, device="cuda"), c(gates)
        ops.lru_scan(c(u), made, c(y), c(lam), s1, *map(c, meta), o1, 8.0, c(yb), True,
                     torch.full((2, T // 32 + n + 1, C), float("nan"), device="cuda"), alone, longest)
        outs.append((s1.cpu(), o1.cpu().float()))
        # only the one-launch form leaves the gates as they are
        assert torch.equal(made.cpu(), gates) == (alone and one_launch(T, n, longest))
        # fp32 sums damped by decays below one: some ten operations per step over the steps that they last; the output and the
        # reference's are each rounded to bf16 once, by up to 2^-8 of the value
        scale = float(s0.abs().max())
        assert float((s1.cpu() - s0).abs().max()) <= 400 * 2.0 ** -24 * scale
        tol = 400 * 2.0 ** -24 * float(o0.float().abs().max()) + (2.0 ** -7 * o0.float().abs() if dtype == torch.bfloat16 else 0)
        off = (o1.cpu().float() - o0.float()).abs()
        assert bool((off <= tol).all()), (alone, longest, float((off - tol).max()))
    for s2, o2 in outs[1:]:
        assert torch.equal(outs[0][0], s2) and torch.equal(outs[0][1], o2)


# one row, threads' and workgroups' edges, 64 experts, all experts, ties, the largest step and one beyond it
@pytest.mark.parametrize("M,E,top,shared", [(1, 16, 2, True), (17, 16, 2, True), (128, 5, 1, False), (129, 64, 8, True), (256, 16, 2, False),
                                            (64, 4, 4, True), (257, 16, 2, True)])
def test_choice_and_work_list(M, E, top, shared):
    g = torch.Generator(device="cuda").manual_seed(M + E)
    W = F = 128
    z = torch.randn(M, E, device="cuda", generator=g)
    z[::3] = (2 * z[::3]).round()  # ties
    S = top + shared
    tiles = -(-M * S // 64) + E + 2

    def lists():
        return [torch.full((n,), -7, dtype=torch.int32, device="cuda") for n in (tiles * 64, tiles, 1)]

    rnd = lambda *s: (torch.randn(*s, device="cuda", generator=g) / s[-1] ** 0.5).bfloat16()  # noqa: E731
    x = rnd(M, W) * W ** 0.5
    ws = [rnd(E, F, W), rnd(E, F, W), rnd(E, W, F)] + ([rnd(F, W), rnd(F, W), rnd(W, F)] if shared else [None] * 3)
    got = []
    for joined in (False, True):
        idx = torch.zeros(M, top, dtype=torch.int32, device="cuda")
        wt = torch.zeros(M, top, device="cuda")
        srt, te, nt = lists()
        if joined:
            aligned = ops.moe_topk_lists(z, idx, wt, srt, te, nt, shared)
            assert aligned == (M <= 256)
        else:
            ops.moe_topk(z, idx, wt)
            aligned = False
        o = torch.zeros(M * S, W, device="cuda")
        ops.moe_grouped(x, idx, wt, *ws, srt, te, nt, torch.zeros(M * S, F, dtype=torch.bfloat16, device="cuda"), o, aligned=aligned)
        got.append((idx, wt, o, te, nt))
    for a, b in zip(*got):
        assert torch.equal(a, b)
