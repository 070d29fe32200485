"""gelu(gate) * up as a GEMM's epilogue (csrc/kernels/gemm_epilogue.h) on every kernel that has one, against float64."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops
from distributed_sse_for_llm_response_amd.ops.reference import gate_up_perm, tile_weight


def check(M, F, K, dev):
    """bf16 inputs, fp32 sums: the result's own rounding (2^-9) and sums of K products in 32 bits ((K + 64) 2^-24 of the largest sum of
    magnitudes, through gelu's slope of at most 1.13 and the other factor)."""
    g = torch.Generator().manual_seed(M + F)
    x = torch.randn(M, K, generator=g).bfloat16()
    w = (torch.randn(2 * F, K, generator=g) / K ** 0.5).bfloat16()
    out = torch.zeros(M, F, dtype=torch.bfloat16, device=dev)
    ops.gemm_gelu(x.to(dev), tile_weight(w[gate_up_perm(F)].contiguous()).to(dev), out)
    z = x.double() @ w.double().t()
    size = x.double().abs() @ w.double().abs().t()
    gate, up = z[:, :F], z[:, F:]
    want = torch.nn.functional.gelu(gate, approximate="tanh") * up
    eps = (K + 64) * 2.0 ** -24 * size
    tol = 2.0 ** -8 * want.abs() + 1.13 * eps[:, :F] * up.abs() + gate.abs() * eps[:, F:] + 2.0 ** -20
    assert ((out.double().cpu() - want).abs() <= tol).all()


def test_gelu_cpu():
    check(3, 64, 512, "cpu")


@pytest.mark.gpu
@pytest.mark.parametrize("F,K", [(8192, 2048), (1024, 1024)])
@pytest.mark.parametrize("M", [1, 8, 9, 17, 48, 64, 65, 128, 150, 256, 257, 400, 1100])
def test_gelu(M, F, K):
    check(M, F, K, "cuda")


# gates far outside exp's range, whose squares overflow: z for the positive ones, zero for the negative ones, in both activations
@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 17, 64, 100, 160, 300])
@pytest.mark.parametrize("act", [ops.gemm_silu, ops.gemm_gelu])
def test_large_gates(M, act):
    F, K = 1024, 1024
    x = torch.zeros(M, K)
    x[:, 0] = 1
    w = torch.zeros(2 * F, K)
    gate = torch.tensor([2.0 ** 10, -2.0 ** 10, 2.0 ** 70, -2.0 ** 70, 2.0 ** 120, -2.0 ** 120, 0.0, float("inf")]).repeat(F // 8)
    w[:F, 0], w[F:, 0] = gate, 0.5
    out = torch.full((M, F), float("nan"), dtype=torch.bfloat16, device="cuda")
    act(x.bfloat16().cuda(), tile_weight(w.bfloat16()[gate_up_perm(F)].contiguous()).cuda(), out)
    want = (gate.clamp_min(0) * 0.5).expand(M, F)
    assert torch.equal(out.float().cpu(), want)
