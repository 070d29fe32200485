"""The shared expert's down product in two slices (moe_grouped with a part more than slots) against the PyTorch reference."""
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


@pytest.fixture
def key(request, monkeypatch):
    monkeypatch.setenv("DSSE_KERNEL_CFG", ops.kernel_cfg_env(**request.param))
    ops.refresh_env()
    yield request.param
    monkeypatch.undo()
    ops.refresh_env()


def _case(M, W, F, Fs, E, top, seed=0):
    g = torch.Generator().manual_seed(M + W + Fs + seed)

    def rnd(*s):
        return (torch.randn(*s, generator=g) / s[-1] ** 0.5).bfloat16()

    x = torch.randn(M, W, generator=g).bfloat16()
    ws = (rnd(E, F, W), rnd(E, F, W), rnd(E, W, F), rnd(Fs, W), rnd(Fs, W), rnd(W, Fs))
    idx = torch.rand(M, E, generator=g).argsort(-1)[:, :top].int().contiguous()
    return x, ws, idx, torch.rand(M, top + 1, generator=g) + 0.25


def _scratch(gpu, M, F, Fs, E, S):
    tiles = -(-M * S // 64) + E + 2
    i32 = dict(dtype=torch.int32, device=gpu)
    return (torch.zeros(tiles * 64, **i32), torch.zeros(tiles, **i32), torch.zeros(1, **i32),
            torch.zeros(M * S, max(F, Fs), dtype=torch.bfloat16, device=gpu))


FORMS = [{"moe_form": 1}, {"moe_form": 2, "moe_once": 1}, {"moe_form": 2, "moe_once": 2}]


# two K steps per slice, the fewest; slices of unlike lengths; row tiles that end inside a list tile and inside a tall tile; column blocks past
# the width; up to 192 rows in the stream, which has three list tiles of the shared expert then
@pytest.mark.parametrize("key,M,W,F,Fs,E,top", [(k, *c) for k in FORMS for c in (
    (1, 128, 128, 256, 2, 2), (65, 320, 192, 320, 3, 2), (192, 448, 128, 1088, 4, 1))] +
    [(k, *c) for k in FORMS[1:] for c in ((257, 192, 128, 448, 2, 1), (700, 576, 320, 576, 8, 2))], indirect=["key"])
def test_two_slices(gpu, key, M, W, F, Fs, E, top):
    x, ws, idx, w = _case(M, W, F, Fs, E, top)
    S = top + 1
    ref = torch.zeros(M * S, W)
    lref.moe_grouped(x, idx, w, *ws, ref)
    c = lambda t: t.to(gpu)  # noqa: E731
    o = torch.full((M * (S + 1), W), float("nan"), device=gpu)
    ops.moe_grouped(c(x), c(idx), c(w), *map(c, ws), *_scratch(gpu, M, F, Fs, E, S), o, parts=S + 1)
    got, ref = o.cpu().view(M, S + 1, W), ref.view(M, S, W)
    # routed parts as ever; the two slices add up to the shared expert's (hidden values rounded to bf16 once, sums in fp32)
    for a, b in ((got[:, :top], ref[:, :top]), (got[:, top] + got[:, S], ref[:, top])):
        assert float((a.double() - b.double()).norm() / b.double().norm()) <= 2.0 ** -8
        assert float((a - b).abs().max()) <= 2.0 ** -5 * float(b.abs().max())
    # and each is the product over its own hidden units
    half = (Fs // 64) // 2 * 64
    cut = [t.clone() for t in ws]
    cut[5][:, half:] = 0
    first = torch.zeros(M * S, W)
    lref.moe_grouped(x, idx, w, *cut, first)
    first = first.view(M, S, W)[:, top]
    assert float((got[:, top].double() - first.double()).norm() / first.double().norm()) <= 2.0 ** -8


@pytest.mark.parametrize("key", [{"moe_form": 3}], indirect=True)
def test_refusals(gpu, key):
    M, W, F, Fs, E, top = 20, 128, 128, 256, 2, 1
    x, ws, idx, w = _case(M, W, F, Fs, E, top)
    c = lambda t: t.to(gpu)  # noqa: E731
    S = top + 1
    args = (c(x), c(idx), c(w), *map(c, ws), *_scratch(gpu, M, F, Fs, E, S))
    assert ops.moe_parts(c(x), top, *map(c, ws), args[-1]) == S  # the register-direct kernels have no slices
    for parts, rows in ((S + 1, S + 1), (S + 2, S + 2), (S, S + 1), (0, S + 1), (S - 1, S - 1)):
        with pytest.raises(RuntimeError):
            ops.moe_grouped(*args, torch.zeros(M * rows, W, device=gpu), parts=parts)


# a long shared expert of one row and of a few hundred; one as long as the routed ones; steps whose tiles fill the chip without; bytes
# that outlast the chain; no shared expert; exact mode
@pytest.mark.parametrize("M,W,F,Fs,E,top,more", [
    (1, 2048, 1408, 2816, 16, 2, 1), (192, 2048, 1408, 2816, 16, 2, 0), (300, 2048, 1408, 2816, 16, 2, 1), (2048, 2048, 1408, 2816, 16, 2, 0),
    (300, 1024, 2048, 2048, 8, 2, 0), (40, 1024, 512, 192, 8, 2, 0)])
def test_rule(gpu, M, W, F, Fs, E, top, more):
    t = lambda *s: torch.empty(s, dtype=torch.bfloat16, device=gpu)  # noqa: E731
    h = t(M * (top + 1), max(F, Fs))
    ws = (t(E, F, W), t(E, F, W), t(E, W, F))
    assert ops.moe_parts(t(M, W), top, *ws, t(Fs, W), t(Fs, W), t(W, Fs), h) == top + 1 + more
    assert ops.moe_parts(t(M, W), top, *ws, None, None, None, h) == top
    f = lambda *s: torch.empty(s, device=gpu)  # noqa: E731
    assert ops.moe_parts(f(M, 128), 2, f(2, 64, 128), f(2, 64, 128), f(2, 128, 64), f(512, 128), f(512, 128), f(128, 512), f(M * 3, 512)) == 3
