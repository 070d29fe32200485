"""Chunks of 16 tokens of the matrix-state recurrence (csrc/kernels/matrix_chunk.hip): decays per key channel, two column tiles per
workgroup, launches in segments; and which calls take them."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops import layers_reference as lref
from distributed_sse_for_llm_response_amd.ops.layers import scan_state_from_plain, scan_state_plain


def i32(x):
    return torch.tensor(x, dtype=torch.int32)


@pytest.mark.parametrize("shift,pitch,two", [(0, 0, False), (4, 4, False), (1, 0, True), (0, 2, True)])
def test_decays_per_channel_take_the_chunks_where_their_rows_are_aligned(shift, pitch, two):
    ops.load_library(required=True)
    T, H, G, D, V = 512, 8, 4, 64, 32
    q, k, v = torch.empty(T, G, D), torch.empty(T, G, D), torch.empty(T, H, V)
    decay = torch.empty(T * (H * D + pitch) + 4)[shift:shift + T * (H * D + pitch)].view(T, -1)[:, :H * D].unflatten(1, (H, D))
    assert torch.ops.dsse.matrix_scan_two_levels(q, k, v, True, T, 2, T // 2, decay) is two


def run(H, G, D, V, ql, mode, bad=None, seed=0):
    """The op against the reference walk: continued and fresh slots, rows outside every sequence that hold NaN.  Error: sums of D
    products and of 16 tokens in fp32 on either side, (D + 64) 2^-24 each of the largest result."""
    g = torch.Generator().manual_seed(seed)
    n, pad = len(ql), 2
    T = sum(ql) + (n + 1) * pad
    qs = [(i + 1) * pad + sum(ql[:i]) for i in range(n)]
    outside = torch.ones(T, dtype=torch.bool)
    for a, m in zip(qs, ql):
        outside[a:a + m] = False
    ctx, slot = [m + (5 if i % 2 == 0 else 0) for i, m in enumerate(ql)], list(range(n, 0, -1))
    q, k = (torch.nn.functional.normalize(torch.randn(T, G, D, generator=g), dim=-1) for _ in range(2))
    v = torch.randn(T, H, V, generator=g)
    if "channel" in mode:
        decay = torch.rand(T, H, D, generator=g) ** 0.2
        decay[pad + 5::13, :, ::3] = 0.0
    else:
        decay = torch.rand(T, H, generator=g) ** 0.2
    beta = torch.rand(T, H, generator=g) if "delta" in mode else None
    if bad is not None:
        {"v": v, "decay": decay}[bad[0]][qs[0] + bad[1], H - 1] = float("nan")
    for t in (q, k, v, decay, beta):
        if t is not None:
            t[outside] = float("nan")
    state0 = torch.randn(n + 1, H, D, V, generator=g)
    st_ref, o_ref = state0.clone(), torch.zeros(T, H, V)
    meta = (i32(qs), i32(ql), i32(ctx), i32(slot))
    lref.matrix_scan(q, k, v, decay, beta, st_ref, *meta, o_ref, 0.5)
    c = lambda t: None if t is None else t.cuda()  # noqa: E731
    st, o = scan_state_from_plain(c(state0)), torch.zeros(T, H, V, device="cuda")
    ops.matrix_scan(c(q), c(k), c(v), c(decay), c(beta), st, *map(c, meta), o, 0.5, max(ql))
    tol = 2 * (D + 64) * 2.0 ** -24
    got = scan_state_plain(st).cpu()
    for a, b in ((o.cpu(), o_ref), (got, st_ref)):
        fine = torch.isfinite(b)
        assert torch.equal(torch.isfinite(a), fine)
        assert (a - b)[fine].abs().max() <= tol * b[fine].abs().max()
    assert torch.equal(got[0], state0[0]) and not o[outside.cuda()].any()   # other slots and rows


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D,V", [(4, 2, 32, 16), (3, 3, 64, 48), (2, 1, 128, 32)])
@pytest.mark.parametrize("mode", ["channel", "delta_channel"])
@pytest.mark.parametrize("ql", [[1, 16, 17, 90, 0, 31], [96], [193, 2], [47, 33, 64]])
def test_decays_per_channel(H, G, D, V, mode, ql):
    run(H, G, D, V, ql, mode, seed=D + len(ql))


@pytest.mark.gpu
@pytest.mark.parametrize("H,D,V,n", [(16, 64, 64, 5), (8, 128, 96, 6), (16, 32, 32, 9)])
@pytest.mark.parametrize("mode", ["channel", "tokens", "delta"])
def test_two_column_tiles_per_workgroup(H, D, V, n, mode):
    assert H * V // 16 * n > 256
    run(H, H // 4, D, V, [100 - 17 * (i % 6) for i in range(n)], mode)


@pytest.mark.gpu
@pytest.mark.parametrize("at", [0, 15, 16, 40])
@pytest.mark.parametrize("bad", ["v", "decay"])
@pytest.mark.parametrize("mode", ["channel", "delta_channel"])
def test_tokens_before_one_that_is_not_finite(mode, bad, at):
    run(4, 2, 64, 32, [130, 70], mode, (bad, at))


@pytest.mark.gpu
@pytest.mark.parametrize("ql,bad", [([2600, 70], None), ([70, 2600], None), ([2600, 70], ("v", 1500))])
def test_segments(ql, bad):
    """64 heads of 128 channels under the delta rule: 72 M workspace floats, taken in segments of 77 chunks."""
    run(64, 1, 128, 16, ql, "delta", bad)
