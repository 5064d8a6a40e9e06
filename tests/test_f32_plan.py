"""Which fp32 kernel and slices a product takes (ops.f32_split_slices), without a GPU."""
import pytest

from operator_amd import ops


@pytest.mark.parametrize("N,K,glu", [(16384, 2048, ops.GELU_TANH), (2048, 2048, 0), (2048, 288, 0), (1072, 2048, 0), (2050, 2048, 0)])
def test_a_prompts_kernel_and_slices_follow_its_padded_rows(N, K, glu):
    for lo in (33, 513, 1537):
        hi = -(-lo // 512) * 512
        plans = {ops.f32_split_slices(ops.f32_plan_rows(M, True), N, K, glu) for M in (lo, lo + 1, hi - 1, hi)}
        assert len(plans) == 1
        (S,) = plans
        assert S is None or 1 <= S <= 8 and (S == 1 or N % 4 == 0)
    assert ops.f32_split_slices(32, N, K, glu) is None   # few rows stream the weights


def test_lines():
    assert ops.f32_split_slices(1024, 16384, 2048, ops.GELU_TANH) == 1
    assert ops.f32_split_rows(962, 16384, 2048, 1, ops.GELU_TANH) == 256
    assert ops.f32_split_slices(512, 2048, 288, 0) is None       # 9 us against 14
    assert ops.f32_split_slices(512, 2048, 8192, 0) is not None  # 161 against 99
