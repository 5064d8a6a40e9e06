"""One to eight rows: the row-streaming kernel (gemm_rows.hip) and the rule that takes products to it."""
import pytest
import torch

from operator_amd import ops

DEV = "cuda"


def _close(y, x, w, exact):
    r, mag = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    tol = w.shape[1] * 2.0 ** -24 * mag + (0 if exact else 2.0 ** -8 * r.abs())   # fp32 sums of K terms; the bf16 result
    assert ((y.double() - r).abs() <= tol).all()


@pytest.mark.gpu
# a wave's quarter of a slice: 32 columns, whole 512-column pieces, a part of the last one, one to eight pieces; rows of W that leave
# the last request and the last workgroup part empty; one row per workgroup
@pytest.mark.parametrize("N,K,S,blocks", [(16, 128, 1, 1), (48, 2048, 1, 7), (1040, 2176, 1, 256), (4096, 4096, 1, 256), (2000, 3584, 2, 96), (272, 5120, 1, 300),
                                          (1008, 14336, 1, 64), (512, 16384, 1, 512), (640, 28672, 4, 40), (2064, 1536, 1, 129)])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8])
def test_rows(M, N, K, S, blocks):
    torch.manual_seed(N + K + M)
    C, pieces = ops.kernels(), -(-K // (2048 * S))
    x, w = torch.randn(M, K, device=DEV).bfloat16(), (torch.randn(N, K, device=DEV) * 0.05).bfloat16()
    p = torch.full((S * M * N,), float("nan"), device=DEV)
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    if pieces * (1 << (M - 1).bit_length()) > 32:   # X does not fit in registers
        with pytest.raises(RuntimeError):
            C.gemm_skinny(x, w, y, p, S, 0, blocks)
        return
    C.gemm_skinny(x, w, None, p, S, 0, blocks)
    s = p.view(S, M, N).double().sum(0)
    _close(s, x, w, True)
    C.gemm_skinny(x, w, y, p, S, 0, blocks)
    _close(y, x, w, False)
    for m in {0, M - 1}:   # a row's bits do not depend on the rows beside it, nor on the workgroups
        q = torch.empty(S * N, device=DEV)
        C.gemm_skinny(x[m:m + 1], w, None, q, S, 0, max(1, blocks // 2))
        assert torch.equal(q.view(S, N), p.view(S, M, N)[:, m])


@pytest.mark.gpu
@pytest.mark.parametrize("N,K,blocks", [(128, 128, 2), (384, 2048, 24), (16512, 512, 257), (1024, 4096, 500), (256, 8192, 100)])
@pytest.mark.parametrize("M", [1, 3, 4, 8])
@pytest.mark.parametrize("act", [ops.SILU, ops.GELU_TANH])
def test_gated_rows(M, N, K, blocks, act):
    torch.manual_seed(N + K + M)
    x = torch.randn(M, K, device=DEV).bfloat16()
    g, u = ((torch.randn(N // 2, K, device=DEV) * K ** -0.5).bfloat16() for _ in range(2))
    y = torch.full((M, N // 2), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.kernels().gemm_skinny(x, ops.interleave_gate_up(g, u), y, None, 1, act, blocks)
    gate, up = x.double() @ g.double().t(), x.double() @ u.double().t()
    f = torch.nn.functional.silu if act == ops.SILU else lambda z: torch.nn.functional.gelu(z, approximate="tanh")
    r = f(gate) * up
    assert ((y.double() - r).abs() <= 2.0 ** -8 * (4 * r.abs() + 1.1 * gate.abs() * up.abs()) + 1e-5).all()   # as in test_skinny_tiles_gpu.py


@pytest.mark.gpu
@pytest.mark.parametrize("K", [2048, 2176, 3584])
def test_odd_values_stay_in_their_row_and_column(K):
    """Lanes past a quarter's end hold zeros of both operands: an infinity or NaN in its first column meets none of them."""
    M, N = 3, 48
    x, w = torch.ones(M, K, device=DEV).bfloat16(), torch.ones(N, K, device=DEV).bfloat16()
    x[1, 0], w[7, 0], w[9, K - 1], w[11, K // 4] = float("inf"), float("inf"), float("nan"), float("-inf")
    y = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    ops.kernels().gemm_skinny(x, w, y, None, 1, 0, 3)
    r = x.float() @ w.float().t()
    assert torch.equal(y.isnan(), r.isnan()) and torch.equal(y[~y.isnan()].float(), r[~r.isnan()].bfloat16().float())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 4096, 4096), (4, 4096, 14336), (8, 4096, 14336), (2, 32000, 2048), (7, 6144, 4096), (2, 4096, 4096), (8, 33920, 6400)])
def test_linear_takes_them_there(M, N, K):
    torch.manual_seed(M)
    x, w = torch.randn(M, K, device=DEV).bfloat16(), (torch.randn(N, K, device=DEV) * 0.05).bfloat16()
    S, _ = ops.rows_plan(M, N, K)
    _close(ops.linear(x, w), x, w, False)
    d = ops.linear(x, w, defer_reduce=True)
    assert isinstance(d, ops.SplitK) and d.S == S   # left in fp32, of one slice too
    _close(d.p[:S * M * N].view(S, M, N).sum(0), x, w, True)
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    assert ops.linear(x, w, out=out) is out
    _close(out, x, w, False)
    wide = torch.full((M, N + 16), float("nan"), dtype=torch.bfloat16, device=DEV)   # rows apart
    if M > 1:   # refused, as by gemm_skinny, which takes whole rows
        with pytest.raises(RuntimeError):
            ops.linear(x, w, out=wide[:, :N])
        assert wide.isnan().all()


@pytest.mark.gpu
def test_norm_takes_one_slab():
    torch.manual_seed(0)
    x, w = torch.randn(2, 4096, device=DEV).bfloat16(), (torch.randn(4096, 4096, device=DEV) * 0.02).bfloat16()
    p = torch.empty(2 * 4096, device=DEV)
    ops.kernels().gemm_skinny(x, w, None, p, 1, 0, 256)
    g, res = torch.rand(4096, device=DEV).bfloat16(), torch.randn(2, 4096, device=DEV).bfloat16()
    a, b = res.clone(), res.clone()
    y = ops.rmsnorm(ops.SplitK(p, 1, 2, 4096), g, 1e-5, residual=a)
    z = ops.rmsnorm(p.view(2, 4096).bfloat16(), g, 1e-5, residual=b)
    assert torch.equal(y, z) and torch.equal(a, b)


def test_rule():
    for M in range(1, 9):
        for N, K in ((4096, 4096), (4096, 14336), (3584, 18944), (8192, 28672), (128256, 8192), (152064, 3584), (32000, 2048), (2144, 4096)):
            for glu in (False, True):
                if glu and N % 128:
                    continue
                plan = ops.rows_plan(M, N, K, glu)
                if plan is None:
                    continue
                S, B = plan
                pieces, mt = -(-K // (2048 * S)), 1 << (M - 1).bit_length()
                assert K % (128 * S) == 0 and pieces <= 8 and pieces * mt <= 32 and (S == 1 or not glu)
                assert (-(-(N // 2 if glu else N) // B) * (2 if glu else 1) + 8) * mt * 64 <= 48 << 10
    assert ops.rows_plan(9, 4096, 4096) is None and ops.rows_plan(1, 2048, 1024) is None and ops.rows_plan(1, 1072, 2048) is None
    assert ops.rows_plan(5, 2048, 2048) is None and ops.rows_plan(4, 2048, 2048) == (1, 256)


def test_short_rows_of_five_and_more_stay_where_they_are_faster():
    """Both sides' times stand at the rule."""
    for M in (5, 8):
        for N, K in ((128256, 1536), (51072, 1536), (152064, 1792), (61440, 2304), (61440, 2560), (16384, 1536), (8192, 2304)):
            assert ops.rows_plan(M, N, K) is None and ops.rows_plan(4, N, K) is not None
        for N, K in ((34432, 2560), (128256, 2048), (128256, 3072), (6144, 1536), (16384, 1792), (20480, 2304), (16384, 2560)):
            assert ops.rows_plan(M, N, K) is not None
        assert ops.rows_plan(M, 98304, 1536, True) is None and ops.rows_plan(M, 20480, 1536, True) is not None
        for N, K in ((14464, 1536), (16256, 1536), (24448, 1536), (16256, 2304), (14464, 2176), (8064, 2176), (8192, 2048), (16256, 2432)):
            assert ops.rows_plan(M, N, K) is None and ops.rows_plan(M, N, K, True) is None and ops.rows_plan(4, N, K) is not None
        for N, K in ((7168, 1536), (14336, 1536), (8064, 2304), (16256, 2048), (14464, 2432), (24448, 2432), (16256, 1664)):   # two slices, a last round less full
            assert ops.rows_plan(M, N, K) is not None


def test_workgroups_do_not_start_in_step():
    """Rows of W 508, 516, 1016 or 1032 KiB apart (gate | up 504, 520, 1008, 1040) have more and smaller workgroups."""
    for N, K, glu in ((16256, 4096, False), (16512, 4096, False), (8128, 8192, False), (11008, 6144, False), (18864, 3584, False), (9440, 14336, False),
                      (16128, 4096, True), (16640, 4096, True), (16128, 8192, True)):
        assert ops.rows_plan(1, N, K, glu) == (1, 768)
    for N, K, glu in ((16384, 4096, False), (16128, 4096, False), (4096, 4096, False), (4096, 14336, False), (16384, 4096, True), (16256, 4096, True)):
        assert ops.rows_plan(1, N, K, glu) == (1, 256)


def test_measured_slices_are_of_products_that_other_kernels_run():
    for k in ops._gemm_table_get():
        if k[0] in ("skinny", "silu"):
            assert ops.rows_plan(*k[1:], k[0] == "silu") is None, k
