"""rmsnorm_fp8 equals quantize_fp8 of the bf16 rmsnorm, byte for byte, from rows and from split-K slabs; the SwiGLU
quantization of long rows equals the unfused kernels."""
import pytest
import torch

from operator_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,hidden,S", [(1, 64, 0), (5, 2048, 1), (64, 4096, 3), (9, 4096, 8), (64, 8192, 4), (3, 8192, 9), (70, 8192, 0), (2, 16384, 2)])
@pytest.mark.parametrize("residual", [False, True])
def test_equals_two_kernels(rows, hidden, S, residual):
    g = torch.Generator(device="cuda").manual_seed(rows + hidden)
    w = torch.randn(hidden, generator=g, device="cuda").bfloat16()
    if S:
        x = ops.SplitK(torch.randn(S * rows * hidden, generator=g, device="cuda"), S, rows, hidden)
    else:
        x = torch.randn(rows, hidden + 8, generator=g, device="cuda").bfloat16()[:, :hidden]   # strided rows
        x[0] = 0
    r = [torch.randn(rows, hidden, generator=torch.Generator(device="cuda").manual_seed(1), device="cuda").bfloat16() if residual else None
         for _ in range(2)]
    q0, s0 = ops.quantize_fp8(ops.rmsnorm(x, w, 1e-5, residual=r[0], out=torch.empty(rows, hidden, dtype=torch.bfloat16, device="cuda")))
    q, s = ops.rmsnorm_fp8(x, w, 1e-5, residual=r[1])
    assert torch.equal(s, s0) and torch.equal(q.view(torch.uint8), q0.view(torch.uint8))
    if residual:
        assert torch.equal(r[0], r[1])


@pytest.mark.parametrize("inter", [8256, 16448, 28672, 32768])
@pytest.mark.parametrize("S", [0, 2, 5])
def test_swiglu_of_long_rows(inter, S):
    g = torch.Generator(device="cuda").manual_seed(inter)
    if S:
        P = torch.randn(S, 3, 2 * inter, generator=g, device="cuda")
        a = P[0].clone()
        for k in range(1, S):
            a += P[k]
        gu, x = a.bfloat16(), ops.SplitK(P.reshape(-1), S, 3, 2 * inter)
    else:
        gu = x = torch.randn(3, 2 * inter, generator=g, device="cuda").bfloat16()
    q, s = ops.silu_quantize_fp8(x, block=64)
    q0, s0 = ops.quantize_fp8(ops.silu_mul(gu, block=64))
    torch.testing.assert_close(s, s0, rtol=1e-6, atol=0)
    # one e4m3fn ulp where the two kernels' silu differ in the last bit of its bf16 rounding
    got, want = q.float(), q0.float()
    assert ((got - want).abs() <= want.abs().clamp(min=2 ** -6) * 2 ** -3 + 1e-12).all() and (got == want).float().mean() > 0.99


def test_long_rows_need_silu_muls_row_stride():
    """Rows past 16384 features come in 16-B aligned strides, as they did when silu_mul read them; shorter ones in any."""
    x = torch.randn(3, 2 * 16448 + 4, device="cuda").bfloat16()
    with pytest.raises(RuntimeError, match="16-B aligned rows"):
        ops.silu_quantize_fp8(x[:, :2 * 16448], block=64)
    y = x[:, :2 * 8192]
    q, s = ops.silu_quantize_fp8(y, block=64)
    q0, s0 = ops.silu_quantize_fp8(y.contiguous(), block=64)
    assert torch.equal(q.view(torch.uint8), q0.view(torch.uint8)) and torch.equal(s, s0)
