"""SiLU and GELU of every gate that bf16 holds, in the epilogues of the dense and of the expert GEMMs, against float64: far below zero the
result is small, not zero."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops.reference import gate_up_perm, tile_weight

pytestmark = pytest.mark.gpu


def _gates(act):
    """Every bf16 number up to 2^100 whose activation is a normal number and whose exponential fp32 holds, and the activation."""
    z = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    z = z[torch.isfinite(z) & (z.abs() < 2.0 ** 100)]
    d = z.double()
    u = d if act == "silu" else 1.5957691216057308 * (d + 0.044715 * d ** 3)
    want = d / (1 + torch.exp(-u))
    keep = (want.abs() > 2.0 ** -124) & (u > -88.6)
    return z[keep], want[keep]


# the result's rounding, and an exponent of up to 128 bits with a rounding or two of its own, 2^-24 of it each
def _check(got, want):
    tol = (2.0 ** -8 + 128 * 2.0 ** -22) * want.abs()
    assert ((got.double() - want).abs() <= tol).all()


@pytest.mark.parametrize("act", ["silu", "gelu"])
@pytest.mark.parametrize("M", [1, 17, 100, 256, 400])
def test_dense(gpu, M, act):
    z, want = _gates(act)
    F, K = -(-z.numel() // 1024) * 1024, 512
    w = torch.zeros(2 * F, K, dtype=torch.bfloat16)
    w[:z.numel(), 0], w[F:, 0] = z, 1
    x = torch.zeros(M, K, dtype=torch.bfloat16)
    x[:, 0] = 1
    out = torch.full((M, F), float("nan"), dtype=torch.bfloat16, device=gpu)
    (ops.gemm_silu if act == "silu" else ops.gemm_gelu)(x.to(gpu), tile_weight(w[gate_up_perm(F)].contiguous()).to(gpu), out)
    for row in {0, M // 2, M - 1}:
        _check(out[row, :z.numel()].cpu(), want)


@pytest.mark.parametrize("form", [1, 2, 3], ids=["stream", "pipeline", "direct"])
def test_experts(gpu, monkeypatch, form):
    monkeypatch.setenv("DSSE_KERNEL_CFG", ops.kernel_cfg_env(moe_form=form))
    ops.refresh_env()
    try:
        z, want = _gates("silu")
        M, W, F = 70, 128, -(-z.numel() // 256) * 256
        x = torch.zeros(M, W, dtype=torch.bfloat16)
        x[:, 0] = 1
        gate, up, down = (torch.zeros(1, *s, dtype=torch.bfloat16) for s in ((F, W), (F, W), (W, F)))
        gate[0, :z.numel(), 0], up[0, :, 0] = z, 1
        h, o = torch.zeros(M, F, dtype=torch.bfloat16, device=gpu), torch.zeros(M, W, device=gpu)
        lists = (torch.zeros(n, dtype=torch.int32, device=gpu) for n in (4 * 64, 4, 1))
        ops.moe_grouped(x.to(gpu), torch.zeros(M, 1, dtype=torch.int32, device=gpu), torch.ones(M, 1, device=gpu), gate.to(gpu), up.to(gpu), down.to(gpu),
                        None, None, None, *lists, h, o)
        for row in (0, M - 1):
            _check(h[row, :z.numel()].cpu(), want)
    finally:
        monkeypatch.undo()
        ops.refresh_env()
