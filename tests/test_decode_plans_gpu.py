"""Decode-bucket projections of shapes without a measured table entry: the chosen tiles and K slices against fp64."""
import pytest
import torch

from operator_amd import ops

pytestmark = pytest.mark.gpu


def _operands(M, N, K):
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).bfloat16().cuda()
    w = (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16().cuda()
    return x, w


# one tile, uneven slices, a plan of each row tile, and gemm_mid's
@pytest.mark.parametrize("M", [64, 128, 192, 256])
@pytest.mark.parametrize("N,K", [(64, 128), (192, 448), (2048, 2048), (3584, 3584), (3584, 18944), (5120, 1408)])
def test_projection(M, N, K):
    x, w = _operands(M, N, K)
    want, mag = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    acc = K * 2.0 ** -24 * mag + 1e-30   # fp32 accumulation of K products, in slices or not
    for defer in (False, True):
        y = ops.linear(x, w, defer_reduce=defer)
        if isinstance(y, ops.SplitK):
            assert ((y.p[:y.S * M * N].view(y.S, M, N).double().sum(0) - want).abs() <= acc).all()
        else:   # ... and one rounding to bf16
            assert ((y.double() - want).abs() <= acc + 2.0 ** -8 * want.abs()).all()


@pytest.mark.parametrize("M", [64, 128, 192, 256])
@pytest.mark.parametrize("N,K", [(128, 128), (1280, 256), (16384, 192), (28672, 128), (37888, 128)])
def test_gate_up(M, N, K):
    x, w = _operands(M, N, K)
    inter = N // 2
    gate, up = ((x.double() @ w.view(-1, 2, 64, K)[:, h].reshape(inter, K).double().t()).bfloat16().double() for h in (0, 1))
    want = (gate * torch.sigmoid(gate)).bfloat16().double() * up
    y = ops.gate_up_silu(x, w, 64).double()
    # each of gate, silu(gate), up and the product may round the other way (2^-8; silu's slope is below 1.1), and a gate
    # near 0 carries its absolute error
    assert ((y - want).abs() <= 5 * 2.0 ** -8 * want.abs() + 2.0 ** -8 * 1.1 * (up * gate).abs() + 1e-6).all()
