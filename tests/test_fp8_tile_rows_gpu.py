"""Tiles of 96, 128 and 160 rows of the fp8 prompt GEMM: the same bits as gemm_fp8, which takes them in tiles of its own, at edges of
tiles, remainders, several rounds and the fewest steps a unit may have."""
import pytest
import torch

from operator_amd import ops

DEV = "cuda"


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,S", [(1, 64, 384, 1), (95, 320, 512, 1), (97, 256, 768, 2), (161, 1088, 384, 1), (321, 4224, 1152, 3),
                                     (885, 6144, 512, 1), (2600, 16384, 384, 1)])
def test_rows(M, N, K, S):
    torch.manual_seed(M + N + K)
    q, sx = ops.quantize_fp8(torch.randn(M, K, device=DEV).bfloat16())
    w, sw = ops.quantize_fp8(torch.randn(N, K, device=DEV).bfloat16())
    C, want = ops.kernels(), ops.linear_fp8((q, sx), w, sw, plan=(64, 64, S))
    slabs = []
    for rows in (96, 128, 160):
        y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
        part = torch.full((S, M, N), float("nan"), device=DEV) if S > 1 else None
        C.gemm_fp8_tile(q, w, sx, sw, y, part, S, rows=rows)
        assert torch.equal(y, want), rows
        if S > 1:
            C.gemm_fp8_tile(q, w, sx, sw, None, part.fill_(float("nan")), S, rows=rows)
            slabs.append(part)
    assert all(torch.equal(p, slabs[0]) for p in slabs)
    exact = (q.double() * sx[:, None]) @ (w.double() * sw[:, None]).t()
    mag = (q.double().abs() * sx[:, None]) @ (w.double().abs() * sw[:, None]).t()
    # one bf16 rounding, fp32 sums of K products and the two scales
    assert ((want.double() - exact).abs() <= 2.0 ** -8 * exact.abs() + (K + 2 + S) * 2.0 ** -24 * mag).all()


def test_rows_that_the_kernel_has():
    for N, K in ((4096, 4096), (57344, 8192), (8192, 28672)):
        for M in (65, 100, 300, 885, 4096, 30000):
            assert ops.fp8_tile_rows(M, N, K, 1)[1] in (96, 128, 160)
    assert [ops.fp8_tile_rows(m, 8192, k, 1)[1] for m, k in ((700, 8192), (1024, 8192), (1200, 28672))] == [96, 128, 160]


def test_small_products_take_the_faster_kernel():
    """A few workgroups: what a kernel needs to start and to store counts (700 rows of 3072 x 2048 13.7 us in tiles of 96 rows, 16.2 on
    gemm_fp8; 128 rows of 4096 x 4096 10.6 on gemm_fp8, 13.3)."""
    for m, n, k in ((700, 3072, 2048), (300, 3584, 4096), (200, 4608, 3584), (1200, 2048, 2048), (150, 3584, 4096)):
        s = ops.fp8_tile_plan(m, n, k)
        assert s == ops._fp8_slices(m, n, k)[2] and ops.fp8_tile_rows(m, n, k, s)[1] == 96
    assert all(ops.fp8_tile_plan(m, 4096, 4096) is None for m in (65, 128))
    assert ops.fp8_tile_plan(65, 10240, 8192) is None and ops.fp8_plan(65, 10240, 8192) == (128, 128, 2)   # 30 us, 36 in tiles of 96 rows
