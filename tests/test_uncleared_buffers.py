"""Prompt passes do not clear the activations that they write whole: whatever the memory held, the logits are the same bit for
bit.  Every layered family, both element types, with prompts that take the small and the large forms of the kernels."""
import pytest
import torch

from distributed_sse_for_llm_response_amd.engine.engine import LLMEngine
from distributed_sse_for_llm_response_amd.models import registry

NAMES = ["muderax-tiny", "surodra-tiny", "dironex-tiny", "murulorn-tiny", "kagorax-tiny", "lobidra-tiny"]
EMPTY = torch.empty


def filled(value):
    def empty(*shape, **kw):
        t = EMPTY(*shape, **kw)
        return t.fill_(value) if t.is_floating_point() else t
    return empty


def passes(device, name, dtype, lens, monkeypatch, value):
    fam, cfg, _ = registry.resolve(name)
    w = registry.load_weights(fam, cfg, None, device=device, seed=0, dtype=dtype)
    r = registry.make_runner(fam, w, num_blocks=sum(-(-n // 32) + 2 for n in lens), max_batch=len(lens),
                             max_model_len=max(lens) + 64, max_prefill_tokens=sum(lens), device=device)
    eng = LLMEngine(r, eos_id=-1)
    eng.watermark = 0
    g = torch.Generator().manual_seed(5)
    toks = [torch.randint(3, cfg.vocab_size, (n,), generator=g).tolist() for n in lens]
    monkeypatch.setattr(torch, "empty", filled(value))
    first = [(str(i), t[:-3], sorted({0, len(t) // 2, len(t) - 4})) for i, t in enumerate(toks)]
    out = [eng.force_step(first), eng.force_step([(str(i), t[-3:], [2]) for i, t in enumerate(toks)])]  # a continued portion
    monkeypatch.setattr(torch, "empty", EMPTY)
    return [o.float().cpu() for o in out]


def same_whatever_was_there(device, name, dtype, lens, monkeypatch):
    zeros, nans = (passes(device, name, dtype, lens, monkeypatch, v) for v in (0.0, float("nan")))
    for a, b in zip(zeros, nans):
        assert torch.isfinite(a).all() and torch.equal(a, b)


@pytest.mark.parametrize("name", NAMES)
def test_reference_ops(name, monkeypatch):
    same_whatever_was_there(torch.device("cpu"), name, torch.float32, [37, 9], monkeypatch)


@pytest.mark.gpu
@pytest.mark.parametrize("lens", [[37, 9], [300, 5, 131]])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("name", NAMES)
def test_kernels(name, dtype, lens, monkeypatch):
    same_whatever_was_there(torch.device("cuda", 0), name, dtype, lens, monkeypatch)
