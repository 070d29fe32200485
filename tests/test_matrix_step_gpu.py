"""Decode rows of the matrix-state recurrence, one wave per 16 columns (matrix_scan_step_kernel in csrc/kernels/matrix_scan.hip),
against the op's reference."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops import layers_reference as lref
from distributed_sse_for_llm_response_amd.ops.layers import scan_state_from_plain, scan_state_plain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,G,D,V", [(4, 2, 16, 16), (3, 3, 32, 80), (2, 1, 64, 64), (2, 2, 128, 112)])
@pytest.mark.parametrize("mode", ["delta", "delta_channel", "channel", "fixed", "plain"])
def test_rows(H, G, D, V, mode):
    """One to three rows per sequence, an empty sequence, fresh and continued slots in reversed order; value tiles that leave
    waves of the last workgroup idle; column slices of wider rows.  Error: sums of D products in fp32 over at most three
    steps, 3 D 2^-24 of the largest result on either side."""
    g = torch.Generator().manual_seed(D + V)
    ql, ctx = [1, 3, 0, 1, 2, 1], [9, 3, 4, 1, 30, 7]
    n, T = len(ql), sum(ql)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32)  # noqa: E731
    meta = (i32([sum(ql[:i]) for i in range(n)]), i32(ql), i32(ctx), i32(list(range(n, 0, -1))))
    wide = torch.randn(T, 2 * G * D + H * V + 4, generator=g)
    wide[:, 1:1 + 2 * G * D] *= D ** -0.5

    def views(t):  # q and k at odd columns, v at a multiple of four
        v0 = 2 * G * D + 4
        return (t[:, 1:1 + G * D].unflatten(1, (G, D)), t[:, 1 + G * D:1 + 2 * G * D].unflatten(1, (G, D)),
                t[:, v0:v0 + H * V].unflatten(1, (H, V)))

    decay = {"delta": torch.rand(T, H, generator=g), "fixed": torch.linspace(0.5, 0.99, H), "plain": None}.get(
        mode, torch.rand(T, H, D, generator=g))
    beta = torch.rand(T, H, generator=g) if "delta" in mode else None
    state0 = torch.randn(n + 1, H, D, V, generator=g)
    st_ref, o_ref = state0.clone(), torch.zeros(T, H, V)
    lref.matrix_scan(*views(wide), decay, beta, st_ref, *meta, o_ref, 0.7)
    c = lambda t: None if t is None else t.cuda()  # noqa: E731
    st, o = scan_state_from_plain(c(state0)), torch.zeros(T, H, V, device="cuda")
    ops.matrix_scan(*views(c(wide)), c(decay), c(beta), st, *map(c, meta), o, 0.7)
    tol = 2 * 3 * D * 2.0 ** -24
    assert (o.cpu() - o_ref).abs().max() <= tol * o_ref.abs().max()
    got = scan_state_plain(st).cpu()
    assert (got - st_ref).abs().max() <= tol * st_ref.abs().max()
    assert torch.equal(got[0], state0[0]) and torch.equal(got[4], state0[4])   # no sequence, the empty one
