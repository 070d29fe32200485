"""A joint layer's sublayers on one stream and on two: the same logits bit for bit, whichever a prompt pass takes, also when the
layers of a pass differ; and the rule is one of the rows."""
import pytest
import torch

from distributed_sse_for_llm_response_amd.engine.engine import LLMEngine
from distributed_sse_for_llm_response_amd.models import registry


def _engine(dev):
    fam, cfg, _ = registry.resolve("kagorax-tiny")
    w = registry.load_weights(fam, cfg, None, device=dev, seed=0, dtype=torch.bfloat16)
    r = registry.make_runner(fam, w, num_blocks=24, max_batch=3, max_model_len=384, max_prefill_tokens=512, device=dev)
    eng = LLMEngine(r, eos_id=-1)
    eng.watermark = 0
    return cfg, r, eng


@pytest.mark.gpu
def test_one_stream_or_two():
    g = torch.Generator().manual_seed(3)
    out = []
    for how in (lambda L, M: False, lambda L, M: True, lambda L, M, n=[0]: n.__setitem__(0, n[0] + 1) or n[0] % 2 == 0):
        cfg, r, eng = _engine(torch.device("cuda", 0))
        r._worth_a_fork = how
        g.manual_seed(3)
        toks = [torch.randint(3, cfg.vocab_size, (n,), generator=g).tolist() for n in (210, 70, 5)]
        passes = [eng.force_step([(str(i), t[:-3], [0, len(t) - 4]) for i, t in enumerate(toks)]),
                  eng.force_step([(str(i), t[-3:], [2]) for i, t in enumerate(toks)])]
        torch.cuda.synchronize()
        out.append([p.float().cpu() for p in passes])
    for other in out[1:]:
        for a, b in zip(out[0], other):
            assert torch.isfinite(a).all() and torch.equal(a, b)


@pytest.mark.gpu
def test_rule_grows_with_the_rows():
    cfg, r, _ = _engine(torch.device("cuda", 0))
    L = next(L for L in cfg.layers if L.mlp is not None)
    worth = [r._worth_a_fork(L, M) for M in (1, 100, 1000, 10 ** 7)]
    assert worth == sorted(worth) and not worth[0] and worth[-1]
