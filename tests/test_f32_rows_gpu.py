"""fp32 products of one to sixteen rows that stream the weights: against 64 bits at every count of rows and pieces, with columns that do not fill the last piece,
rows that are no multiple of anything, four and eight waves and any number of workgroups; what it is refused with; and the rule that takes it."""
import pytest
import torch

from operator_amd import ops
from operator_amd.ops import reference as ref

DEV = "cuda"


def _run(x, w, y, glu, blocks, S=1):
    M, N = x.shape[0], w.shape[0]
    p = torch.full((S * M * N,), float("nan"), device=DEV) if S > 1 else None
    ops.kernels().gemm_f32(x, w, y, glu, partial=p, splits=S, blocks=blocks)
    return y


def _check(x, w, glu, blocks, S=1):
    M, K = x.shape
    N = w.shape[0]
    guard = torch.full((M + 1, N // 2 if glu else N), float("nan"), device=DEV)
    _run(x, w, guard[:M], glu, blocks, S)
    assert guard[M].isnan().all()
    y, r = guard[:M].double(), x.double() @ w.double().t()
    # a lane's chain of at most 32 products, 4 steps over its 16 lanes, at most 8 waves' sums of 4, at most 8 slices: 54 roundings of what the magnitudes amount to
    bound = 54 * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    if not glu:
        assert ((y - r).abs() <= bound).all()
        return
    v, b = (t.view(M, N // 128, 2, 64).transpose(1, 2).reshape(M, 2, N // 2) for t in (r, bound))
    want = ref.silu_mul(torch.cat([v[:, 0], v[:, 1]], 1), None, glu == ops.GELU_TANH)
    gate = ref.silu_mul(torch.cat([v[:, 0], torch.ones_like(v[:, 0])], 1), None, glu == ops.GELU_TANH)
    # the activation's slope is below 1.2; it and the product round in 32 bits behind an exponential of a few ulp
    assert ((y - want).abs() <= 1.2 * b[:, 0] * v[:, 1].abs() + gate.abs() * b[:, 1] + 2.0 ** -20 * want.abs() + 1e-7).all()


@pytest.mark.gpu
@pytest.mark.parametrize("K", [16, 208, 768, 1040, 2048, 3072, 4112, 5120, 6160, 8192])
@pytest.mark.parametrize("M", [1, 2, 3, 5, 8, 9, 16])
def test_rows(M, K):
    torch.manual_seed(M + K)
    x = torch.randn(M, K, device=DEV)
    if not ops.kernels().f32_rows_waves(M, K):
        pytest.skip("too long")
    for N, blocks in ((1, 1), (37, 3), (130, 256), (130, 7)):
        _check(x, torch.randn(N, K, device=DEV) * 0.05, 0, blocks)
    for act in (ops.SILU, ops.GELU_TANH):
        for N, blocks in ((128, 5), (256, 64), (256, 300)):
            _check(x, torch.randn(N, K, device=DEV) * 0.05, act, blocks if M <= 8 or blocks > 5 else 16)


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,S", [(9, 8192, 4), (16, 4096, 2), (13, 6144, 3), (16, 14336, 7), (3, 16384, 8)])
def test_slices(M, K, S):
    torch.manual_seed(M + K)
    for N, blocks in ((4, 1), (36, 5), (132, 64)):
        _check(torch.randn(M, K, device=DEV), torch.randn(N, K, device=DEV) * 0.05, 0, blocks, S)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,glu", [(16, 2048, 8192, 0), (9, 32000, 2048, 0), (12, 16384, 2048, 1), (16, 1024, 2048, 0), (1, 2048, 8192, 0), (8, 2048, 8192, 0), (4, 512, 16384, 0), (3, 16384, 2048, ops.GELU_TANH), (8, 32000, 2048, 0), (6, 2624, 2048, 0)])
def test_products_that_models_have(M, N, K, glu):
    torch.manual_seed(N)
    x, w = torch.randn(M, K, device=DEV), torch.randn(N, K, device=DEV) * 0.05
    S, blocks = ops.f32_rows_plan(M, N, K, glu)
    _check(x, w, glu, blocks, S)
    y = _run(x, w, torch.empty(M, N // 2 if glu else N, device=DEV), glu, blocks, S)
    assert torch.equal(ops.linear_f32(x, w, glu), y)
    if not glu:   # what is infinite or NaN stays with its row, and with its column of W
        x[0, 5], w[7, K - 1] = float("nan"), float("inf")
        z = ops.linear_f32(x, w)
        rest = torch.arange(N, device=DEV) != 7
        assert z[0].isnan().all() and not z[1:, 7].isfinite().any() and torch.equal(z[1:, rest], y[1:, rest])


@pytest.mark.gpu
def test_others_are_refused():
    C, t = ops.kernels(), lambda *s: torch.zeros(*s, device=DEV)   # noqa: E731
    for M, N, K, glu, opt in ((17, 64, 64, 0, {}), (1, 64, 40960, 0, {}), (1, 192, 64, 1, {}), (1, 64, 64, 0, {"rows": 64}), (1, 64, 48, 0, {"splits": 2, "partial": t(128)}), (1, 128, 64, 1, {"splits": 2, "partial": t(256)}), (1, 64, 72, 0, {})):
        with pytest.raises(RuntimeError):
            C.gemm_f32(t(M, K), t(N, K), t(M, N // 2 if glu else N), glu, blocks=4, **opt)


def test_the_rule():
    for a, b in (((1, 2048, 8192, 0), (1, 256)), ((8, 32000, 2048, 0), (1, 768)), ((1, 28672, 4096, 1), (1, 768)), ((1, 8128, 4096, 0), (1, 768)), ((2, 2048, 2048, 0), (1, 256)),
                 ((16, 2048, 8192, 0), (4, 128)), ((9, 16384, 2048, 1), (1, 512)), ((16, 3072, 2048, 0), (1, 256)), ((16, 32000, 2048, 0), (1, 1024)), ((12, 6144, 4096, 0), (2, 256))):
        assert ops.f32_rows_plan(*a) == b, a
    # more rows, longer rows than the registers hold, short rows, few weights, columns that are no multiple of 16
    for a in ((17, 2048, 2048, 0), (8, 2048, 16384, 0), (16, 28672, 4096, 1), (1, 4096, 512, 0), (16, 2048, 768, 0), (1, 16, 2048, 0), (1, 2048, 2056, 0)):
        assert ops.f32_rows_plan(*a) is None, a
    for M in range(1, 17):
        for N in (256, 2048, 32000, 152064):
            for K in range(768, 16384, 1072):
                for glu in (0, 1):
                    n, k = N - N % 128, K - K % 16
                    if (p := ops.f32_rows_plan(M, n, k, glu)) is not None:
                        nw, units = ops.kernels().f32_rows_waves(M, k // p[0]), n // (2 if glu else 1)
                        assert k % (16 * p[0]) == 0 and (-(-units // p[1]) * (2 if glu else 1) + 8) * 16 * nw * (1 << (M - 1).bit_length()) <= 48 << 10
