"""Long sequences of the matrix-state recurrence by chunks of 64 tokens on the matrix cores (csrc/kernels/matrix_chunk.hip),
against the op's reference walk."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops import layers_reference as lref
from distributed_sse_for_llm_response_amd.ops.layers import scan_state_from_plain, scan_state_plain

pytestmark = pytest.mark.gpu


def i32(x):
    return torch.tensor(x, dtype=torch.int32)


@pytest.mark.parametrize("H,G,D,V", [(4, 2, 32, 16), (3, 3, 64, 48), (2, 1, 128, 32)])
@pytest.mark.parametrize("mode", ["delta", "delta_fixed", "tokens", "fixed", "plain"])
@pytest.mark.parametrize("ql,cont", [([1, 64, 65, 130, 0, 3], True), ([96], False), ([193, 2], True)])
def test_chunks_match_the_walk(H, G, D, V, mode, ql, cont):
    """Lengths around the chunk's 64 tokens, an empty and a one-row sequence, continued and fresh slots in reversed order,
    rows outside every sequence that hold NaN (before, between and after them: a chunk of 64 that reaches past its sequence
    may use none of them), column slices of wider rows, decays of exactly zero.  Error: sums of D products and of 64
    tokens in fp32, (D + 64) 2^-24 < 1.2e-5 of the largest result, on either side."""
    g = torch.Generator().manual_seed(3 + D + len(ql))
    n, pad = len(ql), 3
    T = sum(ql) + (n + 1) * pad
    qs = [(i + 1) * pad + sum(ql[:i]) for i in range(n)]
    outside = torch.ones(T, dtype=torch.bool)
    for a, m in zip(qs, ql):
        outside[a:a + m] = False
    ctx = [m + (7 if cont and i % 2 == 0 else 0) for i, m in enumerate(ql)]
    slot = list(range(n, 0, -1))
    wide = torch.randn(T, 2 * G * D + H * V + 3 + 5, generator=g)   # rows of q | k | 3 odd columns | v, to a multiple of 4
    wide = torch.nn.functional.pad(wide, (0, -wide.shape[1] % 4))
    wide[:, G * D:2 * G * D] = torch.nn.functional.normalize(wide[:, G * D:2 * G * D].unflatten(1, (G, D)), dim=-1).flatten(1)
    if "delta" not in mode:
        wide[:, :G * D] *= D ** -0.5
    wide[outside] = float("nan")

    def views(t):
        return (t[:, :G * D].unflatten(1, (G, D)), t[:, G * D:2 * G * D].unflatten(1, (G, D)),
                t[:, 2 * G * D + 3:2 * G * D + 3 + H * V].unflatten(1, (H, V)))

    decay = None
    if mode in ("delta", "tokens"):
        decay = torch.rand(T, H, generator=g) ** 0.2
        decay[pad + 5::17] = 0.0
        decay[outside] = float("nan")
    elif mode != "plain":
        decay = torch.linspace(0.5, 0.999, H)
    beta = torch.rand(T, H, generator=g) if "delta" in mode else None
    if beta is not None:
        beta[outside] = float("nan")
    state0 = torch.randn(n + 1, H, D, V, generator=g)
    st_ref, o_ref = state0.clone(), torch.zeros(T, H, V)
    lref.matrix_scan(*views(wide), decay, beta, st_ref, i32(qs), i32(ql), i32(ctx), i32(slot), o_ref, 0.5)
    c = lambda t: None if t is None else t.cuda()  # noqa: E731
    st, o = scan_state_from_plain(c(state0)), torch.zeros(T, H, V, device="cuda")
    ops.matrix_scan(*views(c(wide)), c(decay), c(beta), st, c(i32(qs)), c(i32(ql)), c(i32(ctx)), c(i32(slot)), o, 0.5, max(ql))
    tol = 2 * (D + 64) * 2.0 ** -24
    assert (o.cpu() - o_ref).abs().max() <= tol * o_ref.abs().max()
    got = scan_state_plain(st).cpu()
    assert (got - st_ref).abs().max() <= tol * st_ref.abs().max()
    assert torch.equal(got[0], state0[0]) and not o[outside.cuda()].any()   # other slots and rows


@pytest.mark.parametrize("delta", [False, True])
def test_the_longest_length_only_chooses_the_form(delta):
    """Sequences that are longer than the caller says: those that the workspace has no room for are walked."""
    g = torch.Generator().manual_seed(11)
    ql, H, D, V = [300, 7, 449], 2, 64, 32
    T, qs = sum(ql), [0, 300, 307]
    q, k, v = (torch.randn(T, H, w, generator=g) * D ** -0.5 for w in (D, D, V))
    decay, beta = torch.rand(T, H, generator=g) ** 0.2, torch.rand(T, H, generator=g) if delta else None
    state0 = torch.randn(3, H, D, V, generator=g)
    st_ref, o_ref = state0.clone(), torch.zeros(T, H, V)
    meta = (i32(qs), i32(ql), i32([m + 1 for m in ql]), i32([2, 0, 1]))
    lref.matrix_scan(q, k, v, decay, beta, st_ref, *meta, o_ref)
    c = lambda t: None if t is None else t.cuda()  # noqa: E731
    for longest in (200, 300, 449, T):
        st, o = scan_state_from_plain(c(state0)), torch.zeros(T, H, V, device="cuda")
        ops.matrix_scan(c(q), c(k), c(v), c(decay), c(beta), st, *map(c, meta), o, 1.0, longest)
        tol = 2 * (D + 64) * 2.0 ** -24   # as above
        assert (o.cpu() - o_ref).abs().max() <= tol * o_ref.abs().max()
        assert (scan_state_plain(st).cpu() - st_ref).abs().max() <= tol * st_ref.abs().max()


@pytest.mark.parametrize("delta", [False, True])
@pytest.mark.parametrize("what", ["q", "k", "v", "inf", "decay", "beta"])
@pytest.mark.parametrize("at", [0, 5, 17, 63, 64, 100])
def test_tokens_before_one_that_is_not_finite(delta, what, at):
    """What a token that is not finite reaches is what the walk lets it reach: later tokens (of one value column, of a head
    group, or its own output alone), never an earlier one."""
    if what == "beta" and not delta:
        return
    g = torch.Generator().manual_seed(at)
    ql, H, G, D, V = [130, 70], 4, 2, 64, 32
    T, qs = sum(ql), [0, 130]
    q, k, v = (torch.randn(T, h, w, generator=g) * D ** -0.5 for h, w in ((G, D), (G, D), (H, V)))
    decay, beta = 0.5 + 0.5 * torch.rand(T, H, generator=g), torch.rand(T, H, generator=g) if delta else None
    if what in ("q", "k"):
        {"q": q, "k": k}[what][at, 1, 3] = float("nan")
    elif what in ("v", "inf"):
        v[at, 1, 9] = float("nan" if what == "v" else "inf")
    else:
        {"decay": decay, "beta": beta}[what][at, 2] = float("nan")
    state0 = torch.randn(2, H, D, V, generator=g)
    st_ref, o_ref = state0.clone(), torch.zeros(T, H, V)
    meta = (i32(qs), i32(ql), i32([m + 1 for m in ql]), i32([1, 0]))
    lref.matrix_scan(q, k, v, decay, beta, st_ref, *meta, o_ref)
    c = lambda t: None if t is None else t.cuda()  # noqa: E731
    st, o = scan_state_from_plain(c(state0)), torch.zeros(T, H, V, device="cuda")
    ops.matrix_scan(c(q), c(k), c(v), c(decay), c(beta), st, *map(c, meta), o, 1.0, T)
    tol = 2 * (D + 64) * 2.0 ** -24   # as above
    for got, ref in ((o.cpu(), o_ref), (scan_state_plain(st).cpu(), st_ref)):
        fine = torch.isfinite(ref)
        assert torch.equal(torch.isfinite(got), fine)
        assert (got - ref)[fine].abs().max() <= tol * ref[fine].abs().max()
