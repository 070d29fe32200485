"""Mixed steps of the layered families: the output projections' parts, many times a step's rows, are not cleared, and whatever the
memory held the logits are the same bit for bit -- with an idle slot among the decode rows and a prompt portion that goes on."""
import pytest
import torch

from distributed_sse_for_llm_response_amd.engine.model_runner import PrefillSeq
from distributed_sse_for_llm_response_amd.models import registry

NAMES = ["muderax-tiny", "surodra-tiny", "dironex-tiny", "murulorn-tiny", "kagorax-tiny", "lobidra-tiny"]
EMPTY, ZEROS = torch.empty, torch.zeros


def _runner(device, name, dtype):
    fam, cfg, _ = registry.resolve(name)
    w = registry.load_weights(fam, cfg, None, device=device, seed=0, dtype=dtype)
    return cfg, registry.make_runner(fam, w, num_blocks=24, max_batch=4, max_model_len=160, max_prefill_tokens=256, device=device)


@pytest.mark.parametrize("name", NAMES)
def test_parts_are_not_cleared(name, monkeypatch):
    _, r = _runner(torch.device("cpu"), name, torch.float32)
    cleared = []
    monkeypatch.setattr(torch, "zeros", lambda *a, **kw: cleared.append(ZEROS(*a, **kw)) or cleared[-1])
    d = r._buffers(40)
    monkeypatch.setattr(torch, "zeros", ZEROS)
    ptrs = {t.data_ptr() for t in cleared}
    assert d["y"].numel() == r._part_rows(40) * r.cfg.width
    for key in ("y", "y2", "ym"):
        assert key not in d or d[key].data_ptr() not in ptrs, key


def _mixed(device, name, dtype, value, monkeypatch):
    cfg, r = _runner(device, name, dtype)
    g = torch.Generator().manual_seed(9)
    toks = torch.randint(3, cfg.vocab_size, (4, 100), generator=g).tolist()
    for s in range(4):
        r.block_tables[s, :4] = torch.arange(4 * s, 4 * s + 4, dtype=torch.int32)
    seq = lambda s, a, b, last: PrefillSeq(slot=s, tokens=toks[s][a:b], start_pos=a, block_table=list(range(4 * s, 4 * s + 4)), last_chunk=last)  # noqa: E731
    r.prefill([seq(0, 0, 40, False), seq(2, 0, 7, False), seq(3, 0, 11, False)], ring_row=0)
    r.active[:3] = torch.tensor([1, 0, 1], dtype=torch.int32)
    ids, pos = [toks[0][40], 0, toks[2][7], 0], [40, 0, 7, 0]

    def empty(*shape, **kw):
        t = EMPTY(*shape, **kw)
        return t.fill_(value) if t.is_floating_point() else t

    out = []
    monkeypatch.setattr(torch, "empty", empty)
    for a, b in ((11, 47), (47, 90)):
        r.ids.copy_(torch.tensor(ids, dtype=torch.int32))
        r.positions.copy_(torch.tensor(pos, dtype=torch.int32))
        r.mixed(4, [seq(3, a, b, b == 90)], ring_row=0)
        out.append(r.logits[[0, 2]].float().cpu())
    monkeypatch.setattr(torch, "empty", EMPTY)
    return out


def _same(device, name, dtype, monkeypatch):
    for a, b in zip(*(_mixed(device, name, dtype, v, monkeypatch) for v in (0.0, float("nan")))):
        assert torch.isfinite(a).all() and torch.equal(a, b)


@pytest.mark.parametrize("name", NAMES)
def test_reference_ops(name, monkeypatch):
    _same(torch.device("cpu"), name, torch.float32, monkeypatch)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("name", NAMES)
def test_kernels(name, dtype, monkeypatch):
    _same(torch.device("cuda", 0), name, dtype, monkeypatch)
