"""SiLU and GELU of every gate that bf16 holds, in the epilogues of the dense GEMMs, against float64: far below zero the
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
