"""The page-sharing form of latent attention for prompt portions (latent_tile.hip) against the PyTorch reference, at the
edges of its column tiles, pages, windows and page-id chunks."""
import math

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


def near(out, ref):
    """Every (row, head) by itself: a wrong column, key or window edge is one of them.  Query vectors, weights and results are
    rounded to bf16 (2^-9 each at most); a rounded query moves a score by some 2^-9 |q||k| / sqrt(D) of it, which the softmax
    passes on: 2^-6 bounds the three together.  One wrong key of n changes a row by some n^-1/2: 2 % of 2100 keys."""
    diff, size = (out.cpu().double() - ref.double()).norm(dim=-1), ref.double().norm(dim=-1)
    assert float((diff / size).max()) <= 2.0 ** -6


# heads that fill eight column tiles exactly, leave some empty, need a second workgroup and are single columns; portions that
# start inside a page, of one row, and behind more than 64 pages; windows of one key, of a page and its neighbours
@pytest.mark.parametrize("H,rk,window", [(32, 512, 10 ** 6), (16, 512, 33), (9, 512, 1), (5, 256, 10 ** 6), (40, 256, 32),
                                         (24, 128, 31), (64, 128, 10 ** 6), (16, 128, 2050)])
def test_prompt_portions(gpu, H, rk, window):
    portions(gpu, H, rk, window, [(0, 70), (31, 1), (64, 33), (2100, 19), (5, 3)], ops.latent_tile_rows(H, rk, 64))


@pytest.mark.parametrize("H,rk,rows", [(33, 512, 1), (16, 128, 1), (9, 256, 1), (8, 256, 2), (5, 128, 2), (4, 128, 4), (1, 512, 4)])
def test_short_prompts(gpu, H, rk, rows):
    """No key further than the second page and few rows: the one-wave form, as many heads side by side as there are."""
    seqs = [(0, 64), (31, 1), (32, 32), (5, 3), (0, 9)]
    assert ops.latent_tile_rows(H, rk, 64, 64, 109) == rows
    assert ops.latent_tile_rows(H, rk, 64, 65, 109) == ops.latent_tile_rows(H, rk, 64, 64, 16384 // H + 1) \
        == ops.latent_tile_rows(H, rk, 64)
    portions(gpu, H, rk, 10 ** 6, seqs, rows)


def portions(gpu, H, rk, window, seqs, rows):
    dn, dr = 24, 64
    g = torch.Generator().manual_seed(H + rk)
    pages = [-(-(s + n) // 32) for s, n in seqs]
    bt = torch.zeros(len(seqs), max(pages), dtype=torch.int32)
    order = torch.randperm(sum(pages) + 2, generator=g)
    qs, at, o = [], 0, 0
    for i, k in enumerate(pages):
        bt[i, :k] = order[at:at + k]
        at += k
        qs.append(o)
        o += seqs[i][1]
    T, ql, ctx = o, [n for _, n in seqs], [s + n for s, n in seqs]
    cache = torch.randn(sum(pages) + 2, 32, rk + dr, generator=g).bfloat16()
    k = torch.arange(32)
    vt = torch.zeros(cache.shape[0], rk, 32, dtype=torch.bfloat16)
    vt[:, :, 8 * ((k & 15) >> 2) + 4 * (k >> 4) + (k & 3)] = cache[:, :, :rk].transpose(1, 2)
    q = torch.randn(T, H, dn + dr, generator=g).bfloat16()
    q_abs = torch.randn(T, H, rk, generator=g) / 4
    rope = torch.randn(max(ctx) + 1, dr // 2, 2, generator=g)
    items = [(i, t) for i in range(len(seqs)) for t in range(-(-ql[i] // rows))]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32)  # noqa: E731
    meta = [i32(x) for x in (qs, ql, ctx, [i for i, _ in items], [t for _, t in items])]
    scale = 1.0 / math.sqrt(dn + dr)
    ref = torch.zeros(T, H, rk)
    lref.latent_attention(q, q_abs, cache, bt, *meta, rope, ref, window, scale, rows, vt)
    out = torch.full((T, H, rk), float("nan"), dtype=torch.bfloat16, device=gpu)
    ops.latent_attention(q.to(gpu), q_abs.to(gpu), cache.to(gpu), bt.to(gpu), *(m.to(gpu) for m in meta), rope.to(gpu), out,
                         window, scale, rows, vt.to(gpu), 16 // rows)
    near(out, ref)
