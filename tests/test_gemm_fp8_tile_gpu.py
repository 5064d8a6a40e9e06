"""gemm_fp8_tile (128 x 256 e4m3fn tiles, K slices): tails, one to several units per workgroup, slices by the reduce pass
and by the consumer, and the plan that chooses it, against float64; gemm_fp8 gives the same bits."""
import pytest
import torch

from operator_amd import ops

pytestmark = pytest.mark.gpu


def _operands(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    q = torch.randn(M, K, generator=g, device="cuda").to(torch.float8_e4m3fn)
    w = torch.randn(N, K, generator=g, device="cuda").to(torch.float8_e4m3fn)
    sx, sw = (torch.rand(n, generator=g, device="cuda") + 0.5 for n in (M, N))
    a, b = q.double() * sx[:, None].double(), w.double() * sw[:, None].double()
    return q, sx, w, sw, a @ b.t(), a.abs() @ b.abs().t()


def _check(y, want, mag, K):
    """One bf16 rounding (2^-8 of the result), fp32 accumulation of K products and the two scales."""
    assert ((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + (K + 2) * 2.0 ** -24 * mag).all()


@pytest.mark.parametrize("M,N,K,S", [
    (1, 16, 384, 1), (128, 256, 512, 1), (129, 272, 896, 2), (300, 1040, 1152, 3), (127, 528, 6144, 16), (700, 16384, 384, 1),
    (2300, 8208, 640, 1), (385, 4160, 1536, 4)])
def test_gemm_fp8_tile(M, N, K, S):
    q, sx, w, sw, want, mag = _operands(M, N, K)
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    part = torch.full((S, M, N), float("nan"), device="cuda") if S > 1 else None
    ops.kernels().gemm_fp8_tile(q, w, sx, sw, y, part, S)
    _check(y, want, mag, K)
    if N % 64 == 0:
        assert torch.equal(y, ops.linear_fp8((q, sx), w, sw, plan=(64, 64, S)))
    if S > 1:
        part.fill_(float("nan"))
        ops.kernels().gemm_fp8_tile(q, w, sx, sw, None, part, S)
        assert ((part.double().sum(0) - want).abs() <= (K + S + 2) * 2.0 ** -24 * mag).all()


@pytest.mark.parametrize("M", [1, 64, 100, 256, 257, 1000])
@pytest.mark.parametrize("N,K", [(64, 256), (192, 1536), (4096, 4096), (10240, 2048)])
def test_planned(M, N, K):
    q, sx, w, sw, want, mag = _operands(M, N, K)
    for defer in (False, True):
        y = ops.linear_fp8((q, sx), w, sw, defer_reduce=defer)
        if isinstance(y, ops.SplitK):
            y = y.p[:y.S * M * N].view(y.S, M, N).sum(0)
        _check(y, want, mag, K + 16)
        same = ops.linear_fp8((q, sx), w, sw, plan=(128, 64, ops.fp8_plan(M, N, K)[2]))
        assert defer or torch.equal(y, same)


def test_infinite_scale_stays_in_its_row():
    q, sx, w, sw, want, mag = _operands(200, 512, 1024)
    sx[70] = float("inf")
    y = torch.empty(200, 512, dtype=torch.bfloat16, device="cuda")
    ops.kernels().gemm_fp8_tile(q, w, sx, sw, y, None, 1)
    keep = torch.arange(200, device="cuda") != 70
    _check(y[keep], want[keep], mag[keep], 1024)
    assert not y[70].isfinite().any()
