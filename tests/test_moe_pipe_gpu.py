"""The pipelined expert GEMMs (moe_pipe.hip) against the PyTorch reference, at the sizes where their tiling changes."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops import layers_reference as lref

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    ops.load_library(required=True)
    return torch.device("cuda", 0)


@pytest.fixture(params=[1, 2], ids=["once", "plain"])
def pipe(request, monkeypatch):
    # steps and experts this small would take other forms
    monkeypatch.setenv("DSSE_KERNEL_CFG", ops.kernel_cfg_env(moe_form=2, moe_once=request.param))
    ops.refresh_env()
    yield
    monkeypatch.undo()
    ops.refresh_env()


# rows of expert 0 sit on both sides of a 64-row list tile and of the 128-, 192- and 256-row tiles; two K steps and odd
# counts of them, fewer and more than the column blocks whose first steps differ; output widths that end inside a column block; no shared expert, one expert, and a work list of more than
# 256 tiles (the list's chunks beyond those held in registers)
@pytest.mark.parametrize("M,W,F,Fs,E,top,first,gated", [
    (128, 128, 128, 128, 2, 2, 64, True), (130, 320, 192, 448, 3, 2, 65, True), (257, 128, 448, 128, 2, 1, 129, True),
    (400, 192, 128, 0, 4, 2, 193, True), (513, 576, 320, 192, 3, 1, 257, True), (300, 128, 128, 0, 1, 1, 300, True),
    (300, 128, 128, 128, 300, 1, 0, True), (700, 256, 192, 0, 3, 1, 256, False), (1100, 512, 128, 0, 2, 1, 1025, False),
    (200, 576, 448, 320, 8, 2, 40, True), (193, 1088, 192, 0, 4, 1, 65, True), (210, 192, 1088, 0, 5, 2, 64, False), (194, 2112, 128, 0, 2, 1, 130, True)])
@pytest.mark.parametrize("weight_input", [False, True])
def test_pipelined_experts(gpu, pipe, M, W, F, Fs, E, top, first, gated, weight_input):
    g = torch.Generator().manual_seed(M + W + F)

    def rnd(*s):
        return (torch.randn(*s, generator=g) / s[-1] ** 0.5).bfloat16()

    x = torch.randn(M, W, generator=g).bfloat16()
    gate, up, down = rnd(E, F, W) if gated else None, rnd(E, F, W), rnd(E, W, F)
    sh = (rnd(Fs, W), rnd(Fs, W), rnd(W, Fs)) if Fs else (None, None, None)
    S = top + (1 if Fs else 0)
    # `first` rows choose expert 0 first, the others begin elsewhere; further choices are the next experts
    start = torch.randint(0, max(1, E - 1), (M,), generator=g) + 1
    start[torch.randperm(M, generator=g)[:first]] = 0
    idx = ((start[:, None] + torch.arange(top)) % E).int()
    w = torch.rand(M, S, generator=g) + 0.25
    ref = torch.zeros(M * S, W)
    lref.moe_grouped(x, idx, w, gate, up, down, *sh, ref, weight_input)
    tiles = -(-M * S // 64) + E + 2
    c = lambda t: None if t is None else t.to(gpu)  # noqa: E731
    o = torch.full((M * S, W), float("nan"), device=gpu)
    ops.moe_grouped(c(x), c(idx), c(w), c(gate), c(up), c(down), *(c(t) for t in sh),
                    torch.zeros(tiles * 64, dtype=torch.int32, device=gpu), torch.zeros(tiles, dtype=torch.int32, device=gpu),
                    torch.zeros(1, dtype=torch.int32, device=gpu),
                    torch.zeros(M * S, max(F, Fs), dtype=torch.bfloat16, device=gpu), o, weight_input)
    # every hidden value is rounded to bf16 once, by at most 2^-8 of itself; the sums are fp32
    err = (o.cpu().double() - ref.double()).norm() / ref.double().norm()
    assert float(err) <= 2.0 ** -8
    assert float((o.cpu() - ref).abs().max()) <= 2.0 ** -5 * float(ref.abs().max())


# Tiles cut over K: two and more pieces of two K steps and odd ones, every height of a row tile, a shared expert, experts without a gate, a walk
# that starts in the middle, 257 tiles (a whole round and one tile), and once by the rule itself (33 K steps).  The list's counters are zero again
# afterwards: a second call on the same list gives the same bits.
@pytest.mark.parametrize("M,W,F,Fs,E,top,first,gated,cut", [
    (70, 256, 256, 0, 2, 1, 64, True, 2), (130, 448, 320, 448, 3, 2, 65, True, 3), (300, 1088, 192, 0, 4, 1, 193, True, 8), (513, 576, 320, 192, 3, 1, 257, True, 4),
    (700, 512, 256, 0, 3, 1, 256, False, 4), (257, 512, 128, 0, 257, 1, 1, True, 4), (200, 2112, 256, 320, 2, 2, 40, True, 0)])
@pytest.mark.parametrize("once", [1, 2], ids=["once", "plain"])
def test_cut_tiles(gpu, monkeypatch, M, W, F, Fs, E, top, first, gated, cut, once):
    monkeypatch.setenv("DSSE_KERNEL_CFG", ops.kernel_cfg_env(moe_form=2, moe_once=once, moe_cut=cut))
    ops.refresh_env()
    try:
        g = torch.Generator().manual_seed(M + W + F)

        def rnd(*s):
            return (torch.randn(*s, generator=g) / s[-1] ** 0.5).bfloat16()

        x = torch.randn(M, W, generator=g).bfloat16()
        gate, up, down = rnd(E, F, W) if gated else None, rnd(E, F, W), rnd(E, W, F)
        sh = (rnd(Fs, W), rnd(Fs, W), rnd(W, Fs)) if Fs else (None, None, None)
        S = top + (1 if Fs else 0)
        start = torch.arange(M) % E if E == M else torch.randint(0, max(1, E - 1), (M,), generator=g) + 1
        start[torch.randperm(M, generator=g)[:first]] = 0
        idx = ((start[:, None] + torch.arange(top)) % E).int()
        w = torch.rand(M, S, generator=g) + 0.25
        ref = torch.zeros(M * S, W)
        lref.moe_grouped(x, idx, w, gate, up, down, *sh, ref)
        tiles = -(-M * S // 64) + E + 1  # as few as the operator takes
        c = lambda t: None if t is None else t.to(gpu)  # noqa: E731
        lists = (torch.full((tiles * 64,), 7, dtype=torch.int32, device=gpu), torch.zeros(tiles, dtype=torch.int32, device=gpu),
                 torch.zeros(1, dtype=torch.int32, device=gpu))
        args = (c(x), c(idx), c(w), c(gate), c(up), c(down), *(c(t) for t in sh), *lists)
        outs = []
        for aligned in (False, True):
            o = torch.full((M * S, W), float("nan"), device=gpu)
            ops.moe_grouped(*args, torch.zeros(M * S, max(F, Fs), dtype=torch.bfloat16, device=gpu), o, aligned=aligned)
            outs.append(o.cpu())
            n = int(lists[2])
            assert int(lists[0][n * 64:(n + 1) * 64].abs().sum()) == 0
        assert torch.equal(*outs)
        err = (outs[0].double() - ref.double()).norm() / ref.double().norm()
        assert float(err) <= 2.0 ** -8  # as above: one rounding of the hidden values, fp32 sums
        assert float((outs[0] - ref).abs().max()) <= 2.0 ** -5 * float(ref.abs().max())
    finally:
        monkeypatch.undo()
        ops.refresh_env()


# Down products that the rule itself cuts (32 K steps and more), with a shared expert of so few hidden units that its tiles, the last of some XCDs, stay
# whole; its hidden units in one and in two slices
@pytest.mark.parametrize("M,W,F,Fs,E,top,slices,pieces", [
    (300, 256, 2048, 128, 8, 1, 1, 8), (300, 512, 4096, 512, 8, 2, 1, 1), (300, 512, 4096, 512, 8, 2, 2, 1), (300, 512, 4096, 512, 4, 1, 2, 4)])
@pytest.mark.parametrize("once", [1, 2], ids=["once", "plain"])
def test_down_products_cut_by_the_rule(gpu, monkeypatch, M, W, F, Fs, E, top, slices, pieces, once):
    monkeypatch.setenv("DSSE_KERNEL_CFG", ops.kernel_cfg_env(moe_form=2, moe_once=once))
    ops.refresh_env()
    try:
        g = torch.Generator().manual_seed(M + F)
        c = lambda t: t.to(gpu)  # noqa: E731
        rnd = lambda *s: (torch.randn(*s, generator=g) / s[-1] ** 0.5).bfloat16()  # noqa: E731
        x, gate, up, down, sh = torch.randn(M, W, generator=g).bfloat16(), rnd(E, F, W), rnd(E, F, W), rnd(E, W, F), (rnd(Fs, W), rnd(Fs, W), rnd(W, Fs))
        S, parts = top + 1, top + slices
        idx = ((torch.arange(M)[:, None] + torch.arange(top)) % E).int()
        walks = torch.ops.dsse.moe_pipe_walks(torch.bincount(idx.flatten(), minlength=E).tolist(), W, F, Fs, top, 1, parts)
        assert int(walks[:, 6].max()) == pieces
        w = torch.rand(M, S, generator=g) + 0.25
        ref = torch.zeros(M * S, W)
        lref.moe_grouped(x, idx, w, gate, up, down, *sh, ref)
        tiles = -(-M * S // 64) + E + 1
        o = torch.full((M * parts, W), float("nan"), device=gpu)
        ops.moe_grouped(*(c(t) for t in (x, idx, w, gate, up, down, *sh)), torch.zeros(tiles * 64, dtype=torch.int32, device=gpu),
                        torch.zeros(tiles, dtype=torch.int32, device=gpu), torch.zeros(1, dtype=torch.int32, device=gpu),
                        torch.zeros(M * S, F, dtype=torch.bfloat16, device=gpu), o, parts=parts)
        got, ref = o.cpu().view(M, parts, W), ref.view(M, S, W)
        got = torch.cat([got[:, :top], got[:, top:].sum(1, keepdim=True)], 1)
        for a, b in ((got[:, :top], ref[:, :top]), (got[:, top:], ref[:, top:])):  # as above, the shared expert by itself
            assert float((a.double() - b.double()).norm() / b.double().norm()) <= 2.0 ** -8
            assert float((a - b).abs().max()) <= 2.0 ** -5 * float(b.abs().max())
    finally:
        monkeypatch.undo()
        ops.refresh_env()


# The order of an expert's rows in the work list is whatever its atomics give; any of them gives the same bits, also where the last tiles are cut
# over K: an expert in two row tiles, one of which is among them (by the rule and by force), and both
@pytest.mark.parametrize("M,W,F,E,cut", [(350, 2112, 320, 3, 0), (600, 2048, 256, 2, 0), (700, 512, 384, 2, 2), (3000, 2048, 512, 8, 0)])
def test_bits_do_not_depend_on_the_order_of_the_list(gpu, monkeypatch, M, W, F, E, cut):
    monkeypatch.setenv("DSSE_KERNEL_CFG", ops.kernel_cfg_env(moe_form=2, moe_cut=cut))
    ops.refresh_env()
    try:
        g = torch.Generator().manual_seed(M + F)
        rnd = lambda *s: (torch.randn(*s, generator=g) / s[-1] ** 0.5).bfloat16().to(gpu)  # noqa: E731
        x, gate, up, down = rnd(M, W), rnd(E, F, W), rnd(E, F, W), rnd(E, W, F)
        idx, w = (torch.arange(M)[:, None] % E).int().to(gpu), torch.rand(M, 1, generator=g).to(gpu)
        tiles = -(-M // 64) + E + 1
        lists = (torch.zeros(tiles * 64, dtype=torch.int32, device=gpu), torch.zeros(tiles, dtype=torch.int32, device=gpu), torch.zeros(1, dtype=torch.int32, device=gpu))
        outs = []
        for turn in range(3):
            if turn:  # an order of its own inside every expert
                ids, at = lists[0].cpu(), 0
                for e in range(E):
                    rows = M // E + (e < M % E)
                    ids[at:at + rows] = torch.arange(e, M, E, dtype=torch.int32)[torch.randperm(rows, generator=g)]
                    at += -(-rows // 64) * 64
                lists[0].copy_(ids)
            o = torch.full((M, W), float("nan"), device=gpu)
            h = torch.zeros(M, F, dtype=torch.bfloat16, device=gpu)
            ops.moe_grouped(x, idx, w, gate, up, down, None, None, None, *lists, h, o, aligned=turn > 0)
            outs.append((h.cpu(), o.cpu()))
        for h, o in outs[1:]:
            assert torch.equal(h, outs[0][0]) and torch.equal(o, outs[0][1])
    finally:
        monkeypatch.undo()
        ops.refresh_env()


# 16 K steps are never cut: no workspace; 32 may be
@pytest.mark.parametrize("W,F,cuts", [(1024, 512, False), (2048, 512, True), (1024, 2048, True)])
def test_workspace_only_where_a_tile_may_be_cut(gpu, monkeypatch, W, F, cuts):
    monkeypatch.setenv("DSSE_KERNEL_CFG", ops.kernel_cfg_env(moe_form=2))
    ops.refresh_env()
    try:
        M, E = 300, 4
        z = lambda *s, **k: torch.zeros(*s, device=gpu, **k)  # noqa: E731
        b, i = {"dtype": torch.bfloat16}, {"dtype": torch.int32}
        args = (z(M, W, **b), z(M, 1, **i), z(M, 1), z(E, F, W, **b), z(E, F, W, **b), z(E, W, F, **b), None, None, None, z(10 * 64, **i), z(10, **i), z(1, **i),
                z(M, F, **b), z(M, W))
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        ops.moe_grouped(*args)
        assert (torch.cuda.max_memory_allocated() - before > 0) == cuts
    finally:
        monkeypatch.undo()
        ops.refresh_env()


# results that begin four bytes past a multiple of 16: the same bits, nothing beside them
@pytest.mark.parametrize("shift", [1, 2, 3])
def test_results_of_any_alignment(gpu, monkeypatch, shift):
    monkeypatch.setenv("DSSE_KERNEL_CFG", ops.kernel_cfg_env(moe_form=2))
    ops.refresh_env()
    try:
        M, W, F, E, top = 300, 320, 192, 4, 2
        g = torch.Generator().manual_seed(shift)
        rnd = lambda *s: (torch.randn(*s, generator=g) / s[-1] ** 0.5).bfloat16().to(gpu)  # noqa: E731
        x, gate, up, down = rnd(M, W), rnd(E, F, W), rnd(E, F, W), rnd(E, W, F)
        idx, w = ((torch.arange(M)[:, None] + torch.arange(top)) % E).int().to(gpu), torch.rand(M, top, generator=g).to(gpu)
        n = M * top * W
        bufs = []
        for at in (0, shift):
            tiles = -(-M * top // 64) + E + 1
            lists = (torch.zeros(k, dtype=torch.int32, device=gpu) for k in (tiles * 64, tiles, 1))
            buf = torch.full((n + 8,), float("nan"), device=gpu)
            ops.moe_grouped(x, idx, w, gate, up, down, None, None, None, *lists, torch.zeros(M * top, F, dtype=torch.bfloat16, device=gpu),
                            buf[at:at + n].view(M * top, W))
            assert torch.isnan(buf[:at]).all() and torch.isnan(buf[at + n:]).all()
            bufs.append(buf[at:at + n])
        assert torch.equal(*bufs)
    finally:
        monkeypatch.undo()
        ops.refresh_env()
