"""The fp8 decode GEMM's ring of stages: deeper for narrow tiles of one workgroup per CU and slices of 24 steps or more. Tiles of 128
columns keep three stages: the same bits on either."""
import pytest
import torch

from operator_amd import ops

DEV = "cuda"


# slices of one step, fewer than the deep ring's stages, one less than 24, 24, uneven ones of 24 and 25, many; ragged rows
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,S", [(1, 128, 128, 1), (7, 128, 640, 1), (64, 256, 2944, 1), (64, 256, 3072, 1), (65, 128, 6272, 2), (130, 384, 14336, 4),
                                     (64, 8192, 6144, 2), (64, 8320, 6144, 2)])
def test_rings_give_the_same_bits(M, N, K, S):
    torch.manual_seed(M + N + K)
    q, sx = ops.quantize_fp8(torch.randn(M, K, device=DEV).bfloat16())
    w, sw = ops.quantize_fp8(torch.randn(N, K, device=DEV).bfloat16())
    got = {}
    for bm, bn in ((64, 128), (64, 64), (128, 64)):
        y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
        part = torch.full((S, M, N), float("nan"), device=DEV) if S > 1 else None
        ops.kernels().gemm_fp8(q, w, sx, sw, y, part, S, bn, bm)
        got[bm, bn] = y
    for y in got.values():
        assert torch.equal(y, got[64, 128])
    exact = (q.double() * sx[:, None]) @ (w.double() * sw[:, None]).t()
    mag = (q.double().abs() * sx[:, None]) @ (w.double().abs() * sw[:, None]).t()
    # one bf16 rounding, fp32 sums of K products and the two scales
    assert ((got[64, 64].double() - exact).abs() <= 2.0 ** -8 * exact.abs() + (K + 2 + S) * 2.0 ** -24 * mag).all()


def test_columns_of_few_rows():
    """Up to 64 rows: the narrow tile unless more of them end on one CU; the slices stay."""
    for n, k, cols in ((40960, 8192, 64), (37888, 3584, 64), (57344, 8192, 128), (28672, 4096, 128), (10240, 8192, 64)):
        assert all(ops.fp8_plan(m, n, k) == (64, cols, ops._fp8_slices(m, n, k)[2]) for m in (1, 64))
