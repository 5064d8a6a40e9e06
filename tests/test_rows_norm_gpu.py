"""gemm_rows with the RMSNorm in front of it: rows from bf16 or slabs, with and without a residual, ragged last pieces, against rmsnorm and the
product in float64; and what norm_into leaves to the kernels of its own."""
import pytest
import torch

from operator_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,S,res,kind,blocks", [
    (1, 48, 4096, 1, True, "y", 3), (1, 300, 8192, 4, True, "p", 256), (1, 256, 7296, 0, False, "glu", 5), (2, 64, 4224, 1, True, "p", 64),
    (2, 16, 8192, 0, True, "y", 1), (3, 128, 4096, 2, True, "glu", 17), (4, 1000, 2560, 1, False, "y", 256), (4, 256, 2048, 3, True, "glu", 7),
    (3, 80, 1664, 0, True, "p", 80), (2, 512, 2048, 1, True, "y", 33)])
def test_norm_then_rows(M, N, K, S, res, kind, blocks):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    t = torch.randn(max(S, 1), M, K, generator=g, device="cuda")
    x = t.contiguous() if S else t[0].bfloat16()
    h, nw = torch.randn(M, K, generator=g, device="cuda").bfloat16(), torch.rand(K, generator=g, device="cuda").bfloat16()
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    total = torch.full((M, K), float("nan"), dtype=torch.bfloat16, device="cuda") if res else None
    out = torch.full((M, N // 2 if kind == "glu" else N), float("nan"), dtype=torch.float32 if kind == "p" else torch.bfloat16, device="cuda")
    before = h.clone()
    ops.kernels().gemm_rows_norm(x, S, h if res else None, total, nw, 1e-5, w, *((None, out) if kind == "p" else (out, None)), int(kind == "glu"), blocks)
    want = h.clone()
    xn = ops.rmsnorm(ops.SplitK(x, S, M, K) if S else x, nw, 1e-5, residual=want if res else None)
    assert torch.equal(h, before) and (not res or torch.equal(total, want))
    ref = xn.double() @ w.double().t()
    mag = xn.double().abs() @ w.double().abs().t()
    # the sum of squares in another order moves a normalised value, rounded to bf16 twice, by at most 2^-7 of it, a few of them: a random sum
    tol = 2.0 ** -7 * (xn.double() ** 2 @ w.double().t() ** 2).sqrt() + K * 2.0 ** -24 * mag
    if kind == "glu":
        r = ref.view(M, N // 128, 2, 64)
        gate, up = r[:, :, 0].reshape(M, -1), r[:, :, 1].reshape(M, -1)
        e = tol.view(M, N // 128, 2, 64)
        eg, eu = (e[:, :, i].reshape(M, -1) for i in (0, 1))
        sg = torch.nn.functional.silu(gate)
        ref = sg * up
        tol = (1.1 * eg + 2.0 ** -8 * (gate.abs() + sg.abs())) * up.abs() + (eu + 2.0 ** -8 * up.abs()) * (sg.abs() + 1.1 * eg)
    assert ((out.double() - ref).abs() <= tol + (0 if kind == "p" else 2.0 ** -8 * ref.abs())).all()


def test_what_stays_a_kernel():
    w, nw = torch.randn(4096, 4096, device="cuda").bfloat16(), torch.ones(4096, device="cuda").bfloat16()
    rows = lambda M: torch.randn(M, 4096, device="cuda").bfloat16()  # noqa: E731
    assert ops.norm_into(rows(4), nw, 1e-5, rows(4), w) is not None
    assert ops.norm_into(rows(5), nw, 1e-5, rows(5), w) is None
    assert ops.norm_into(rows(3), nw, 1e-5, rows(3), torch.empty(28672, 4096, dtype=torch.bfloat16, device="cuda"), True) is None
    assert ops.norm_into(rows(1).float(), nw, 1e-5, None, w) is None
    assert ops.norm_into(rows(1), nw, 1e-5, None, w.to(torch.float8_e4m3fn)) is None
    assert ops.norm_into(rows(4)[::2], nw, 1e-5, None, w) is None
    with pytest.raises(RuntimeError):
        h = rows(1)
        ops.kernels().gemm_rows_norm(h, 0, h, h, nw, 1e-5, w, torch.empty_like(h))
