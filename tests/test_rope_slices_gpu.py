"""RoPE and K/V write from the K slices of a split projection: bit for bit what the summed, rounded rows give, for one slice and more
than are loaded together, rows that make whole pages and rows that do not, skipped rows."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,S", [(1, 1), (31, 2), (64, 5), (97, 6), (130, 3)])
@pytest.mark.parametrize("nh,nkv", [(4, 2), (3, 1), (5, 5)])
def test_slices(T, S, nh, nkv):
    g = torch.Generator(device="cuda").manual_seed(T + S)
    width, pages = (nh + 2 * nkv) * 128, T // 32 + 5
    # eighths up to 16: every partial sum is exact, so the order of the slices cannot show
    part = torch.randint(-128, 129, (S, T, width), generator=g, device="cuda").float() / 8
    pos = torch.arange(T, dtype=torch.int32, device="cuda") % 50
    slots = torch.arange(T, dtype=torch.int32, device="cuda") + 64          # whole pages from row 0 on
    if T > 70:
        slots[40:70] = slots[40:70].flip(0)                                   # out of order
        slots[50] = -1
    rope = torch.randn(64, 64, 2, generator=g, device="cuda")
    out = []
    for ns in (0, S):
        qkv = part.sum(0).to(torch.bfloat16) if ns == 0 else torch.full((T, width), float("nan"), device="cuda").to(torch.bfloat16)
        q = torch.zeros(T, nh, 128, dtype=torch.bfloat16, device="cuda")
        kc = torch.zeros(pages, nkv, 32, 128, dtype=torch.bfloat16, device="cuda")
        vc = torch.zeros(pages, nkv, 128, 32, dtype=torch.bfloat16, device="cuda")
        ops.rope_kv_write(qkv, pos, slots, rope, q, kc, vc, nh, nkv, part if ns else None, ns)
        out.append((q, kc, vc))
    for a, b in zip(*out):
        assert torch.equal(a, b)


def test_refused():
    z = lambda *s, dtype=torch.bfloat16: torch.zeros(*s, dtype=dtype, device="cuda")  # noqa: E731
    i = z(2, dtype=torch.int32)
    args = (z(2, 384), i, i, z(4, 64, 2, dtype=torch.float32), z(2, 1, 128), z(1, 1, 32, 128), z(1, 1, 128, 32), 1, 1)
    for part in (None, z(2 * 384, dtype=torch.float32), z(4 * 384)):
        with pytest.raises(RuntimeError):
            ops.rope_kv_write(*args, part, 2)


def test_rows_of_another_width_are_refused():
    z = lambda *s, dtype=torch.bfloat16: torch.zeros(*s, dtype=dtype, device="cuda")  # noqa: E731
    i = z(2, dtype=torch.int32)
    with pytest.raises(RuntimeError):  # one head's worth of columns too few for nh + 2 nkv heads
        ops.rope_kv_write(z(2, 256), i, i, z(4, 64, 2, dtype=torch.float32), z(2, 1, 128), z(1, 1, 32, 128), z(1, 1, 128, 32), 1, 1,
                          z(2, 2, 256, dtype=torch.float32), 2)
