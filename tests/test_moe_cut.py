"""Which K steps the workgroups of the expert GEMM pipeline take (csrc/kernels/moe_cut.h): host code, by the kernel's own rules."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops


def _walks(rows, W, F, Fs, top, product, parts=0, cut=0):
    ops.load_library(required=True)
    return torch.ops.dsse.moe_pipe_walks(rows, W, F, Fs, top, product, parts, cut).tolist()


def _check(walks, steps_r, steps_s, experts):
    """Every tile's pieces hold two K steps or more and make its walk without a gap; returns the counts of pieces."""
    tiles = {}
    for xcd, e, rt, block, sl, piece, of, first, n in walks:
        assert n >= 2, "a piece of fewer steps than the pipeline always runs"
        assert 0 <= piece < of
        tiles.setdefault((e, rt, block, sl), []).append((xcd, piece, of, first, n))
    for (e, rt, block, sl), p in tiles.items():
        p.sort(key=lambda t: t[1])
        assert [t[1] for t in p] == list(range(p[0][2])) and len({t[0] for t in p}) == 1
        assert all(a[3] + a[4] == b[3] for a, b in zip(p, p[1:]))
    for e in {k[0] for k in tiles}:
        for rt, block in {k[1:3] for k in tiles if k[0] == e}:
            walk = sorted((t[3], t[4]) for k, p in tiles.items() if k[:3] == (e, rt, block) for t in p)
            assert walk[0][0] == 0 and sum(n for _, n in walk) == (steps_s if e == experts else steps_r)
    # which of an expert's row tiles holds a row is not fixed, so the sums of a column block have one order in all of them
    for e, block in {(k[0], k[2]) for k in tiles if k[0] < experts}:
        assert len({len(p) for k, p in tiles.items() if (k[0], k[2]) == (e, block)}) == 1
    return {k: len(p) for k, p in tiles.items()}


# a shared expert whose walk is shorter than the pieces of a routed tile, among the last tiles of an XCD: one and two choices a row, slices, a list
# that leaves experts without rows; a step whose last tiles are routed
@pytest.mark.parametrize("M,W,F,Fs,E,top,parts", [
    (300, 256, 2048, 128, 8, 1, 0), (300, 512, 4096, 512, 8, 2, 0), (300, 512, 4096, 512, 8, 2, 4), (1024, 2048, 1408, 2816, 16, 2, 0), (3000, 4096, 3584, 7168, 16, 2, 0),
    (3000, 4096, 3584, 7168, 16, 2, 4), (700, 256, 8192, 256, 4, 1, 3), (350, 2112, 320, 0, 3, 1, 0), (600, 2048, 256, 0, 2, 1, 0)])
@pytest.mark.parametrize("cut", [0, 1, 3, 8])
@pytest.mark.parametrize("uneven", [False, True])
def test_pieces(M, W, F, Fs, E, top, parts, cut, uneven):
    rows = [M * top // E] * E
    if uneven:
        rows = [0, 1] + rows[2:]
    rows[-1] += M * top - sum(rows)
    for product in (0, 1, 2) if not Fs else (0, 1):
        _check(_walks(rows, W, F, Fs, top, product, parts, cut), (F if product == 1 else W) // 64, (Fs if product == 1 else W) // 64, E)


def test_pieces_over_many_sizes():
    g = torch.Generator().manual_seed(7)
    cut = 0
    for _ in range(150):
        r = lambda lo, hi: int(torch.randint(lo, hi, (1,), generator=g))  # noqa: E731
        E, top = r(1, 17), r(1, 3)
        top = min(top, E)
        W, F, Fs = 64 * r(2, 66), 64 * r(2, 130), 64 * r(2, 130) * r(0, 2)
        M = r(1, 2500)
        share = torch.rand(E, generator=g) ** r(1, 4)
        rows = (share / share.sum() * M * top).int().tolist()
        rows[r(0, E)] += M * top - sum(rows)
        S = top + (1 if Fs else 0)
        for product in (0, 1):
            slices = 2 if product and Fs >= 256 and r(0, 2) else 1
            walks = _walks(rows, W, F, Fs, top, product, S + slices - 1)
            cut += any(n > 1 for n in _check(walks, (F if product else W) // 64, (Fs if product else W) // 64, E).values())
    assert cut > 5  # the rule cuts some of them
