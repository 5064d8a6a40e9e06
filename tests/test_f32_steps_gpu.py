"""The fp32 tile GEMM's ring: fewer steps than stages, one more, a half step at the end, plain and gated, whole and in K slices."""
import pytest
import torch

from operator_amd import ops

DEV = "cuda"


@pytest.mark.gpu
@pytest.mark.parametrize("K", [16, 32, 48, 64, 96, 112, 128, 144, 272])
@pytest.mark.parametrize("S", [1, 2])
def test_steps(K, S):
    torch.manual_seed(K)
    M, N = 70, 256
    x, w = torch.randn(M, K, device=DEV), torch.randn(N, K, device=DEV)
    y, part = torch.full((M, N), float("nan"), device=DEV), torch.full((S, M, N), float("nan"), device=DEV)
    ops.kernels().gemm_f32(x, w, y, False, partial=part, splits=S)
    r, mag = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    assert ((y.double() - r).abs() <= (K + S) * 2.0 ** -24 * mag).all()   # K products and sums of 32 bits
    g, u = torch.randn(N // 2, K, device=DEV) * K ** -0.5, torch.randn(N // 2, K, device=DEV)
    z = torch.full((M, N // 2), float("nan"), device=DEV)
    ops.kernels().gemm_f32(x, ops.interleave_gate_up(g, u), z, ops.SILU, partial=part, splits=S)
    a, b = x.double() @ g.double().t(), x.double() @ u.double().t()
    ma, mb = x.double().abs() @ g.double().abs().t(), x.double().abs() @ u.double().abs().t()
    act = torch.nn.functional.silu(a)
    # the sums' errors through the activation (slope below 1.1) and the product, and 8 roundings of its own
    tol = 2.0 ** -24 * ((K + S) * (1.1 * ma * b.abs() + act.abs() * mb) + 8 * (act * b).abs()) + 1e-9
    assert ((z.double() - act * b).abs() <= tol).all()
