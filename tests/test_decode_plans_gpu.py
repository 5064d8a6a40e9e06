"""Decode-bucket projections of shapes without a measured table entry: the chosen tiles and K slices against a
float32 product."""
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
    want = x.float() @ w.float().t()
    for defer in (False, True):
        y = ops.linear(x, w, defer_reduce=defer)
        if isinstance(y, ops.SplitK):
            y = y.p[:y.S * M * N].view(y.S, M, N).sum(0)
        # rows of unit-variance sums: fp32 accumulation, one rounding to bf16 (2^-9 of |y| < 6)
        assert (y.float() - want).abs().max() < 6 * 2 ** -8


@pytest.mark.parametrize("M", [64, 128, 192, 256])
@pytest.mark.parametrize("N,K", [(128, 128), (1280, 256), (16384, 192), (28672, 128), (37888, 128)])
def test_gate_up(M, N, K):
    x, w = _operands(M, N, K)
    inter = N // 2
    want = x.float() @ w.float().t()
    want = want.bfloat16().float().view(M, N // 128, 2, 64)
    gate = torch.nn.functional.silu(want[:, :, 0]).bfloat16().float()
    want = (gate * want[:, :, 1]).reshape(M, inter)
    y = ops.gate_up_silu(x, w, 64).float()
    # gate, up, silu(gate) and the product are rounded: an ulp of gate or up on either side of a rounding is 2^-8
    # of them, |gate|, |up| < 6
    assert (y - want).abs().max() < 36 * 2 ** -7
    assert (y - want).abs().mean() < 2 ** -8
