"""The 256-row expert tiles (gemm_tile.hip, routed): every row's own scale on the gated operands, where a workgroup walks
several tiles and the scales of the next one are requested while this one's rows are still being multiplied."""
import pytest
import torch

from operator_amd import ops

DEV = "cuda"


@pytest.mark.gpu
# tiles x column tiles: one workgroup each, a few rounds of 256, a last round of one; K: the shortest loop (2 steps), an odd one
@pytest.mark.parametrize("tiles,inter,K", [(1, 64, 128), (3, 128, 192), (40, 1024, 128), (33, 1024, 320), (257, 128, 128)])
def test_scales_of_expert_tiles(tiles, inter, K):
    torch.manual_seed(tiles + K)
    E, rows = 3, 256 * tiles
    x = torch.randn(rows, K, device=DEV).bfloat16()
    w = (torch.randn(E, 2 * inter, K, device=DEV) * 0.05).bfloat16()
    wgu = torch.stack([ops.interleave_gate_up(v[:inter], v[inter:]) for v in w])
    expert = torch.randint(0, E, (tiles,), device=DEV)
    gtab = torch.cat([torch.tensor([tiles], device=DEV), expert]).int()
    scale = torch.rand(rows, device=DEV) + 0.1
    y = torch.full((rows, inter), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.kernels().moe_gemm_tile(x, wgu, y, gtab, scale, True)
    gu = torch.cat([x[256 * i:256 * (i + 1)].double() @ w[e].double().t() for i, e in enumerate(expert.tolist())]) * scale[:, None].double()
    gate, up = gu[:, :inter], gu[:, inter:]
    r = torch.nn.functional.silu(gate) * up
    # bf16 rounds to 2^-8 of a value: up, the activation and the product move r by that much each, the gate by its own 2^-8 times
    # the activation's slope (below 1.1) times up; second-order terms are within the fourth r, fp32 sums of K terms far below
    tol = 2.0 ** -8 * (4 * r.abs() + 1.1 * gate.abs() * up.abs()) + 1e-5
    assert ((y.double() - r).abs() <= tol).all()
