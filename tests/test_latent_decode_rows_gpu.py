"""Latent decode attention: every instantiated row size, heads on either side of the two workgroup shapes, and contexts at the edges
of a tile, of two and of the tiles held ahead."""
import pytest
import torch

from operator_amd.ops import decoder as dec

DEV = "cuda"


@pytest.mark.gpu
@pytest.mark.parametrize("H", [3, 16, 17, 40])
@pytest.mark.parametrize("rank,rot", [(96, 32), (128, 64), (192, 64), (256, 32), (336, 48), (400, 48), (448, 64), (512, 64), (576, 64)])
def test_rows(H, rank, rot):
    torch.manual_seed(H + rank)
    L = dec.LatentLayout(H, 64, rot, 64, 128, rank)
    P, lens = 16, [0, 1, 15, 63, 64, 65, 127, 128, 129, 191, 193, 257, 400]
    B, mp = len(lens), 25
    bt = torch.randperm(B * mp + 1, device=DEV)[:B * mp].int().view(B, mp)
    cache = torch.full((B * mp + 1, 1, P, L.ck), float("inf"), device=DEV).bfloat16()   # what no token wrote stays out
    q = torch.randn(B, H, L.ck, device=DEV).bfloat16()
    want = torch.zeros(B, H, L.rp, dtype=torch.float64, device=DEV)
    scale = L.ck ** -0.5
    for b, n in enumerate(lens):
        if not n:
            continue
        rows = torch.randn(n, L.ck, device=DEV).bfloat16()
        for t in range(0, n, P):
            cache[bt[b, t // P], 0, :min(P, n - t)] = rows[t:t + P]
        p = torch.softmax(q[b].double() @ rows.double().t() * scale, -1)
        want[b] = p @ rows[:, :L.rp].double()
    for splits in (1, 3):
        o = dec.attn_latent_decode(q, cache, bt, torch.tensor(lens, dtype=torch.int32, device=DEV), L, scale, splits)
        # weights are rounded to bf16 (2^-9 of each, and they add up to 1), the result once more; rows are about 1, up to 5
        assert ((o.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -8 * 5).all()
