"""The exact mode's expert GEMMs (LDS-DMA strips) against 64 bits: one row and one more than a sub-tile, a tile and its next, an
expert without rows and one with all, widths that end inside a workgroup's columns and inside four chunks, experts with and without a
gate, weights on the inputs, a shared expert of another width."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops

pytestmark = pytest.mark.gpu


def _act(a, b):
    return torch.nn.functional.silu(a) * b if a is not None else torch.relu(b) ** 2


def _reference(x, ti, tw, gate, up, down, shared, weight_in):
    d = lambda t: None if t is None else t.double()  # noqa: E731
    M, top = ti.shape
    out = torch.zeros(M, top + (shared is not None), x.shape[1], dtype=torch.float64, device=x.device)
    mul = lambda a, w: None if w is None else a @ w.T.contiguous()  # noqa: E731
    for k in range(top):
        for e in range(up.shape[0]):
            r = (ti[:, k] == e).nonzero()[:, 0]
            if len(r):
                w = d(tw[r, k])[:, None]
                xi = d(x[r]) * (w if weight_in else 1.0)
                y = mul(_act(mul(xi, None if gate is None else d(gate[e])), mul(xi, d(up[e]))), d(down[e]))
                out[r, k] = y if weight_in else w * y
    if shared is not None:
        sg, su, sd = map(d, shared)
        y = mul(_act(mul(d(x), sg), mul(d(x), su)), sd)
        out[:, top] = y if tw.shape[1] == top else d(tw[:, top])[:, None] * y
    return out


@pytest.mark.parametrize("M", [1, 15, 17, 64, 65, 130])
@pytest.mark.parametrize("W,F,Fs,gated,weight_in", [(128, 128, 0, True, False), (160, 224, 96, True, True), (288, 160, 416, True, False),
                                                    (192, 128, 0, False, False)])
def test_against_float64(M, W, F, Fs, gated, weight_in):
    g = torch.Generator(device="cuda").manual_seed(M + W)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    E, top = 5, 2
    x = rn(M, W)
    gate, up, down = rn(E, F, W) / W ** .5 if gated else None, rn(E, F, W) / W ** .5, rn(E, W, F) / F ** .5
    shared = (rn(Fs, W) / W ** .5, rn(Fs, W) / W ** .5, rn(W, Fs) / Fs ** .5) if Fs else None
    # expert 1 has every row, expert 4 none
    ti = torch.stack([torch.ones(M, dtype=torch.int32), torch.tensor([0, 2, 3], dtype=torch.int32)[torch.arange(M) % 3]], 1).cuda()
    S = top + (Fs > 0)
    tw = torch.rand(M, S if weight_in else top, generator=g, device="cuda") + 0.5
    tiles = -(-M * S // 64) + E + 2
    lists = [torch.zeros(n, dtype=torch.int32, device="cuda") for n in (tiles * 64, tiles, 1)]
    h, o = torch.full((M * S, max(F, Fs) + 4), float("nan"), device="cuda"), torch.full((M * S, W), float("nan"), device="cuda")
    ops.moe_grouped(x, ti, tw, gate, up, down, *(shared or (None, None, None)), *lists, h, o, weight_in)
    ref = _reference(x, ti, tw, gate, up, down, shared, weight_in)
    got = o.view(M, S, W).double()
    # three products in a row, each a random walk of up to max(W, F, Fs) roundings of 2^-24 of a partial sum, and the square's doubling
    bound = 8 * max(W, F, Fs) ** 0.5 * 2.0 ** -24
    for k in range(S):
        assert float((got[:, k] - ref[:, k]).norm() / ref[:, k].norm()) <= bound
