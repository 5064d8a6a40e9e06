"""Few rows: the weight tiles of a workgroup (gemm_skinny.hip skinny_tiles) change what it reads, not the order of a sum."""
import pytest
import torch

from operator_amd import ops

DEV = "cuda"


@pytest.mark.gpu
# features: one tile, an odd number of tiles (only one fits), two and four per workgroup, several rounds; K steps of a wave: one, a
# remainder, groups of 8 and 16; rows at the edges of the two X tiles
@pytest.mark.parametrize("N,K,S", [(16, 128, 1), (48, 1152, 1), (8224, 384, 1), (4096, 1024, 2), (4096, 2304, 2), (8192, 2048, 4), (70016, 2048, 1),
                                   (131072, 256, 1), (8192, 8192, 1)])   # the last: W rows 16 KiB apart, up to 12 X rows on fewer tiles
@pytest.mark.parametrize("M", [1, 5, 16, 17, 32])
def test_rows_are_the_same_beside_others(M, N, K, S):
    torch.manual_seed(N + K + M)
    C = ops.kernels()
    x = torch.randn(32, K, device=DEV).bfloat16()
    w = (torch.randn(N, K, device=DEV) * 0.05).bfloat16()

    def product(rows):
        if S > 1:
            C.gemm_skinny(x[rows], w, None, p := torch.full((S, rows.stop - rows.start, N), float("nan"), device=DEV), S, 0)
            return p
        C.gemm_skinny(x[rows], w, y := torch.full((rows.stop - rows.start, N), float("nan"), dtype=torch.bfloat16, device=DEV), None, 1, 0)
        return y[None]

    y = product(slice(0, M))
    for i in (0, M - 1):   # one row runs on other tiles: the same bits
        assert torch.equal(y[:, i], product(slice(i, i + 1))[:, 0])
    r = x[:M].double() @ w.double().t()
    mag = x[:M].double().abs() @ w.double().abs().t()
    tol = K * 2.0 ** -24 * mag + (2.0 ** -8 * r.abs() if S == 1 else 0)   # fp32 sums of K terms; the bf16 result
    assert ((y.double().sum(0) - r).abs() <= tol).all()


@pytest.mark.gpu
@pytest.mark.parametrize("N,K", [(128, 128), (384, 1152), (16512, 512), (28672, 1024)])
@pytest.mark.parametrize("M", [1, 3, 16, 17, 32])
def test_gated_rows_are_the_same_beside_others(M, N, K):
    torch.manual_seed(N + K + M)
    C = ops.kernels()
    x = torch.randn(32, K, device=DEV).bfloat16()
    g, u = ((torch.randn(N // 2, K, device=DEV) * 0.05).bfloat16() for _ in range(2))
    w = ops.interleave_gate_up(g, u)

    def product(rows):
        C.gemm_skinny(x[rows], w, y := torch.full((rows.stop - rows.start, N // 2), float("nan"), dtype=torch.bfloat16, device=DEV), None, 1, ops.SILU)
        return y

    y = product(slice(0, M))
    for i in (0, M - 1):
        assert torch.equal(y[i], product(slice(i, i + 1))[0])
    gate, up = x[:M].double() @ g.double().t(), x[:M].double() @ u.double().t()
    r = torch.nn.functional.silu(gate) * up
    # bf16 rounds to 2^-8 of a value: up, the activation and the product move r by that much each, the gate by its own 2^-8 times the
    # activation's slope (below 1.1) times up; second-order terms are within the fourth r, fp32 sums far below
    assert ((y.double() - r).abs() <= 2.0 ** -8 * (4 * r.abs() + 1.1 * gate.abs() * up.abs()) + 1e-5).all()
