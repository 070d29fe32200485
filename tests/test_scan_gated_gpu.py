"""Decode rows of a matrix-state recurrence with the head's gated norm in the same launch against both apart: idle sequences, a first
step, a sequence of two rows, one tile of columns and the widest head, all kinds of decay, both element types; and what is refused."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops

pytestmark = pytest.mark.gpu


def _inputs(H, G, D, V, decays, delta):
    g = torch.Generator(device="cuda").manual_seed(D + V)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    ql, ctx = [1, 0, 2, 1], [1, 9, 30, 700]
    T = sum(ql)
    wide = rn(T, 2 * G * D + 2 * H * V + 8)
    q, k = wide[:, :G * D].unflatten(1, (G, D)) / D ** 0.5, wide[:, G * D:2 * G * D].unflatten(1, (G, D))
    v, gate = wide[:, 2 * G * D:2 * G * D + H * V].unflatten(1, (H, V)), wide[:, 2 * G * D + H * V:2 * G * D + 2 * H * V]
    decay = {0: None, 1: torch.rand(H, generator=g, device="cuda"), 2: torch.rand(T, H, generator=g, device="cuda"),
             3: torch.rand(T, H, D, generator=g, device="cuda")}[decays]
    beta = torch.rand(T, H, generator=g, device="cuda") if delta else None
    return q, k, v, decay, beta, rn(5, H, D, V), i32([0, 1, 1, 3]), i32(ql), i32(ctx), i32([2, 0, 4, 1]), gate, rn(V)


@pytest.mark.parametrize("H,G,D,V,decays,delta", [(2, 1, 16, 16, 0, True), (3, 3, 32, 48, 1, False), (4, 2, 64, 64, 2, True),
                                                  (4, 4, 128, 128, 3, False), (2, 2, 128, 256, 2, True)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind", [0, 1])
def test_step_and_norm_together(H, G, D, V, decays, delta, dtype, kind):
    q, k, v, decay, beta, state, qs, ql, ctx, slot, gate, w = _inputs(H, G, D, V, decays, delta)
    for weight in (w, None):
        s0, s1, o = state.clone(), state.clone(), torch.zeros(4, H, V, device="cuda")
        want, got = (torch.zeros(4, H * V, dtype=dtype, device="cuda") for _ in range(2))
        ops.matrix_scan(q, k, v, decay, beta, s0, qs, ql, ctx, slot, o, 0.7)
        ops.gated_head_norm(o, weight, gate, 1e-5, want, kind)
        assert ops.matrix_scan_gated(q, k, v, decay, beta, s1, qs, ql, ctx, slot, weight, gate, 1e-5, got, 0.7, kind)
        # a S + k u, fused or not as the compiler likes: a rounding of either term, twice for the sequence of two rows
        assert float((s0 - s1).abs().max()) <= 4 * 2.0 ** -24 * float(s0.abs().max())
        # the read-out of a state that close; its squares summed in another order, a quotient and an exponential: a few roundings, in bf16 one more
        tol = 2.0 ** -8 if dtype == torch.bfloat16 else 30 * 2.0 ** -24
        assert float((want.double() - got.double()).abs().max()) <= tol * max(1.0, float(want.double().abs().max()))


def test_refused():
    for H, G, D, V in ((2, 2, 24, 32), (2, 2, 32, 24), (1, 1, 32, 272)):
        q, k, v, decay, beta, state, qs, ql, ctx, slot, gate, w = _inputs(H, G, D, V, 0, False)
        out = torch.full((4, H * V), 7.0, device="cuda")
        assert not ops.matrix_scan_gated(q, k, v, decay, beta, state, qs, ql, ctx, slot, w, gate, 1e-5, out)
        assert (out == 7.0).all()
    q, k, v, decay, beta, state, qs, ql, ctx, slot, gate, w = _inputs(2, 2, 32, 32, 0, False)
    one = torch.tensor([4], dtype=torch.int32, device="cuda")  # a prompt portion
    assert not ops.matrix_scan_gated(q, k, v, decay, beta, state, one - 4, one, one, one - 4, w, gate, 1e-5, torch.zeros(4, 64, device="cuda"))
