"""fp32 prefill attention: the two wave groups that take 32-key tiles in turn, and their meeting at the end."""
import pytest
import torch

from operator_amd.ops import decoder as dec

DEV = "cuda"
pytestmark = pytest.mark.gpu


# rows and keys at the edges of a tile, of a pair of tiles and of the 64 query rows; the first group alone, the second behind the window or
# past the end; a shared prefix whose end is inside either group's tile
@pytest.mark.parametrize("lens,prefix", [([1, 31, 32, 33], 0), ([63, 64, 65, 97, 128, 129], 0), ([5, 40], 20), ([5, 70], 33), ([1, 1], 64)])
@pytest.mark.parametrize("D,Dv,window", [(64, 64, 0), (128, 128, 33), (128, 96, 0), (256, 208, 70)])
def test_groups_meet(lens, prefix, D, Dv, window):
    torch.manual_seed(sum(lens) + D + prefix)
    H, G, T = 4, 2, sum(lens)
    L = dec.HeadLayout(H, G, D, Dv)
    q, k, v = (3 * torch.randn(T, h, d, device=DEV) for h, d in ((H, D), (G, D), (G, Dv)))
    pk, pv = (3 * torch.randn(prefix, G, d, device=DEV) for d in (D, Dv))
    gate = torch.rand(T, H, device=DEV)
    pfx = (pk, pv, torch.full((len(lens),), prefix, dtype=torch.int32, device=DEV), [prefix] * len(lens)) if prefix else None
    o = dec.attn_gd_prefill(q, k, v, lens, L, D ** -0.5, prefix=pfx, window=window, gate=gate)[:, :H * Dv].view(T, H, Dv)
    a = 0
    for n in lens:
        kk, vv = (torch.cat([p, t[a:a + n]]).repeat_interleave(H // G, 1).double() for p, t in ((pk, k), (pv, v)))
        s = (q[a:a + n].double().transpose(0, 1) @ kk.permute(1, 2, 0).contiguous()) * D ** -0.5
        i, j = torch.arange(prefix, prefix + n, device=DEV)[:, None], torch.arange(prefix + n, device=DEV)[None]
        hidden = (j > i) | ((i - j >= window) if window else False)
        p = torch.softmax(s.masked_fill(hidden, float("-inf")), -1)
        r = (p @ vv.transpose(0, 1).contiguous()).transpose(0, 1) * gate[a:a + n, :, None].double()
        # scores of up to some 100 carry D 2^-24 of their terms into the weights; values are about 3
        torch.testing.assert_close(o[a:a + n].double(), r, atol=2e-4, rtol=2e-5)
        a += n


# few rows on two wave groups, many on one, alone and with a gate, a shared prefix and a window: a prompt's numbers are the same bits in either
# form. Head sizes that fill an instantiation's blocks and ones that do not
@pytest.mark.parametrize("D,Dv", [(64, 64), (40, 24), (128, 128), (128, 96), (80, 70), (256, 256), (192, 128)])
@pytest.mark.parametrize("prefix,window", [(0, 0), (33, 0), (0, 50)])
def test_packing_does_not_matter(D, Dv, prefix, window):
    torch.manual_seed(D + prefix)
    H, G = 8, 2
    L = dec.HeadLayout(H, G, D, Dv)
    dk, dv = L.pads
    mine = [200, 65, 33, 1]   # each alone: 200 to 33 rows on two groups, or one (256)
    rest = [40] * 70 + [300] * 7   # behind them: more workgroups than two groups are used for
    lens = mine + rest
    T = sum(lens)
    q, k, v = (torch.randn(T, h, d, device=DEV) for h, d in ((H, dk), (G, dk), (G, dv)))
    v[100, 1, 3] = float("inf")   # of the first prompt, in the path of its own for such values
    pk, pv = (torch.randn(prefix, G, d, device=DEV) for d in (dk, dv))
    gate = torch.rand(T, H, device=DEV)

    def run(a, b, ls):
        pfx = (pk, pv, torch.full((len(ls),), prefix, dtype=torch.int32, device=DEV), [prefix] * len(ls)) if prefix else None
        return dec.attn_gd_prefill(q[a:b], k[a:b], v[a:b], ls, L, D ** -0.5, prefix=pfx, window=window, gate=gate[a:b])

    packed, a = run(0, T, lens), 0
    for n in mine:
        assert torch.equal(run(a, a + n, [n]).nan_to_num(nan=7.0), packed[a:a + n].nan_to_num(nan=7.0))
        a += n
