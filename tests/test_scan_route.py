"""Which form a long recurrence without the delta rule takes: the kernels' one decision (scan_two_levels in
csrc/kernels/matrix_chunk.hip), on host tensors -- it looks at shapes, row pitches and addresses."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops


def two_levels(T, H, G, D, V, seqs=1, channels=False, pitch=0, shift=0, longest=None):
    ops.load_library(required=True)
    width = 2 * G * D + H * V + pitch
    wide = torch.empty(T * width + 4)[shift:shift + T * width].view(T, width)
    q, k = (wide[:, c:c + G * D].unflatten(1, (G, D)) for c in (0, G * D))
    v = wide[:, 2 * G * D:2 * G * D + H * V].unflatten(1, (H, V))
    return torch.ops.dsse.matrix_scan_two_levels(q, k, v, channels, T, seqs, longest or -(-T // seqs))


@pytest.mark.parametrize("D", [32, 64, 128])
def test_chunks_where_they_take_the_shape(D):
    assert not two_levels(512, 16, 8, D, 64)
    assert not two_levels(4096, 16, 8, D, 64)
    assert not two_levels(4096, 16, 8, D, 64, pitch=4)


@pytest.mark.parametrize("kw", [dict(channels=True), dict(pitch=1), dict(pitch=2), dict(shift=1), dict(D=48), dict(V=24),
                                dict(T=200000, H=32, seqs=8)])
def test_two_levels_where_chunks_are_refused(kw):
    """Decays per key channel that the question comes without, rows that do not keep 16-byte alignment, other widths, more rows times
    heads than the chunks take."""
    a = dict(T=512, H=16, G=8, D=64, V=64)
    a.update(kw)
    assert two_levels(**a)
    a["T"] = 255
    assert not two_levels(**a)   # short groups are walked


def test_two_levels_for_one_long_sequence_of_few_columns():
    assert two_levels(2048, 2, 2, 128, 128) and two_levels(2048, 4, 4, 64, 64) and two_levels(4096, 4, 2, 32, 32)
    assert not two_levels(800, 2, 2, 128, 128) and not two_levels(1000, 4, 4, 64, 64) and not two_levels(2048, 4, 2, 32, 32)
    assert not two_levels(2048, 4, 4, 128, 128)


# widths that the chunks refuse (the lists will be asked for), widths that they take, and a group too short for two levels
@pytest.mark.gpu
@pytest.mark.parametrize("dim,vdim,rows,made", [(10, 7, 256, True), (32, 16, 256, False), (10, 7, 255, False)])
def test_chunk_lists_are_ready_before_the_first_launch(dim, vdim, rows, made, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    import test_surodra as S
    from distributed_sse_for_llm_response_amd.engine.model_runner import PrefillSeq

    r = S.Model(S.config([S.ff(S.par(rdim=dim, rvdim=vdim)), S.ret(dim=dim, vdim=vdim)]), "cuda", max_tokens=512).runner
    assert len(r._plain_scans) == 2
    asked = []
    real = type(r)._scan_lists
    monkeypatch.setattr(type(r), "_scan_lists", lambda self, g: asked.append("ck" in g) or real(self, g))
    monkeypatch.setattr(type(r), "_layers", lambda self, *a, layers=type(r)._layers, **k: asked.append("layers") or layers(self, *a, **k))
    r.prefill([PrefillSeq(slot=0, tokens=S.toks(rows), start_pos=0, block_table=list(range(8)), last_chunk=True)], ring_row=0)
    # made once, before the layers; found by both of them
    assert asked == ([False, "layers", True, True] if made else ["layers"])


# the costs of both forms (csrc/kernels/matrix_chunk.hip): one and many sequences, few column blocks and many, where the two were measured
# 10 % and more apart; a decode step, and one long portion among portions of one row
@pytest.mark.parametrize("H,D,V,lens,delta,channels,chunks", [
    (16, 128, 128, [64], True, False, True), (16, 128, 128, [2048], False, False, True), (16, 128, 128, [8], True, False, False),
    (8, 128, 128, [200], False, True, True), (16, 64, 16, [32] * 64, True, False, False), (16, 64, 16, [24] * 128, True, True, False),
    (2, 128, 32, [17] * 64, True, False, False), (8, 128, 16, [16] * 64, True, False, False), (16, 128, 32, [64] * 32, True, False, True),
    (4, 64, 16, [128] * 64, True, False, True), (16, 64, 16, [300] * 8, False, False, True), (16, 32, 16, [24] * 128, False, False, False),
    (16, 64, 16, [1] * 60 + [40], True, False, True), (16, 128, 128, [1] * 64, True, False, False)])
def test_walk_or_chunks(H, D, V, lens, delta, channels, chunks):
    ops.load_library(required=True)
    T = sum(lens)
    q, k, v = torch.empty(T, H, D), torch.empty(T, H, D), torch.empty(T, H, V)
    decay = torch.empty(T, H, D) if channels else None
    assert torch.ops.dsse.matrix_scan_by_chunks(q, k, v, delta, channels, T, len(lens), max(lens), decay) is chunks
