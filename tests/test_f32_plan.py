"""Which fp32 kernel and slices a product takes (ops.f32_split_slices), without a GPU."""
import os
import subprocess

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


@pytest.mark.parametrize("N,K,glu", [(16384, 2048, ops.GELU_TANH), (2048, 8192, 0), (3200, 1376, ops.SILU), (8064, 960, ops.SILU), (384, 6048, ops.SILU),
                                     (2912, 560, 0), (2050, 2048, 0), (704, 688, 0), (1024, 96, ops.SILU)])
def test_sums_are_no_longer_than_on_the_fp32_instruction(N, K, glu):
    for M in (33, 40, 64, 100, 200, 512, 1024, 1536, 2048, 4096):
        S = ops.f32_split_slices(M, N, K, glu)
        assert S is None or S >= ops.kernels().gemm_f32_splits(M, N, K, glu)


def test_the_fewest_rows_of_a_plan_are_no_slower():
    """Prompts of 33 rows have the plan of 512: where the split kernel is slower for them in every number of slices, it is not taken."""
    assert ops.f32_split_slices(512, 2912, 560, 0) is None and ops.f32_split_slices(512, 620, 3024, 0) is None   # 33 rows: 11 us against 18, 15 and 21
    assert ops.f32_split_slices(512, 6144, 2048, 0) >= 2      # in one slice 46 us against 56, in two 33
    assert ops.f32_split_slices(512, 2050, 2048, 0) is None   # has no slices: 47 and 56
    assert ops.f32_split_slices(300, 2050, 2048, 0) is None and ops.f32_split_slices(500, 2050, 2048, 0) == 1   # no prompts: rows as they are


def test_the_split_kernels_loads_stay_in_their_rows(tmp_path):
    """Every piece that the kernel requests, two behind the last of a row and of a slice among them, for all K up to 200 and slices up to 8."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    src, exe = tmp_path / "columns.cpp", tmp_path / "columns"
    src.write_text("""
#include <cstdio>
#include "kernels/f32_piece.h"
int main() {
  for (int K = 16; K <= 200; K += 16)
    for (int S = 1; S <= 8; ++S)
      for (int z = 0; z < S; ++z) {
        const int T = (K + 31) / 32, from = z * T / S * 32, to = (z + 1) * T / S * 32;
        for (int k = from; k <= to + 128; k += 32)
          for (int lc = 0; lc < 4; ++lc) {
            const int at = oamd::split_column(k, lc, K);
            if (at < 0 || at + 8 > K || (k + 8 * lc < K && at != k + 8 * lc)) return std::printf("K %d k %d lc %d: %d\\n", K, k, lc, at), 1;
          }
      }
}
""")
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(root, "csrc"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
