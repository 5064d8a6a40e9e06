"""Routed slots in expert segments: one workgroup for few, a workgroup per 1024 slots for many (the line grows with the experts)."""
import pytest
import torch

from operator_amd import ops
from operator_amd.ops import decoder as dec

DEV = "cuda"


# around the line between the two forms, a ragged last workgroup; experts nobody chose, one that everybody did, more of them than slots of a
# workgroup's share
@pytest.mark.gpu
@pytest.mark.parametrize("T,top,E,bm,skew", [(1, 2, 8, 64, 0), (1024, 2, 8, 256, 0), (1025, 2, 8, 256, 0), (2049, 1, 3, 128, 1), (7950, 2, 8, 256, 0),
                                             (3000, 2, 8, 256, 2), (700, 4, 512, 64, 0), (4097, 8, 512, 64, 0), (1589, 2, 8, 64, 0), (1590, 2, 8, 64, 0),
                                             (2741, 1, 3, 128, 1), (1400, 8, 512, 64, 0)])
def test_segments(T, top, E, bm, skew):
    torch.manual_seed(T + E)
    score = torch.randn(T, E, device=DEV)
    if skew:
        score[:, E // 2] += 100.0        # everybody's
        score[:, :E // 2] -= 1000.0      # nobody's
    wt, ids = score.topk(top, -1)
    ids, wt = ids.int(), torch.sigmoid(wt).contiguous()
    rows = dec.expert_rows_bound(T * top, E, bm)
    i32 = dict(dtype=torch.int32, device=DEV)
    pos, src, gtab = torch.full((T, top), -7, **i32), torch.full((rows,), -7, **i32), torch.full((1 + rows // bm,), -7, **i32)
    rs = torch.full((rows,), float("nan"), device=DEV)
    ops.kernels().moe_sort(ids, wt, E, bm, pos, src, rs, gtab)
    counts = torch.bincount(ids.flatten().long(), minlength=E)
    tiles = -(-counts // bm)
    n = int(tiles.sum())
    assert int(gtab[0]) == n
    owner = torch.repeat_interleave(torch.arange(E, device=DEV), tiles)
    assert torch.equal(gtab[1:1 + n].long(), owner)
    p = pos.flatten().long()
    assert p.unique().numel() == T * top and int(p.min()) >= 0 and int(p.max()) < n * bm
    assert torch.equal(owner[p // bm], ids.flatten().long())
    first = (tiles.cumsum(0) - tiles) * bm
    assert (p - first[ids.flatten().long()] < counts[ids.flatten().long()]).all()   # slots in front of the padding
    assert torch.equal(src[p].long(), torch.arange(T * top, device=DEV) // top) and torch.equal(rs[p], wt.flatten())
    pad = torch.ones(n * bm, dtype=torch.bool, device=DEV)
    pad[p] = False
    assert (src[:n * bm][pad] == -1).all() and (rs[:n * bm][pad] == 0).all()
    assert (src[n * bm:] == -7).all() and (gtab[1 + n:] == -7).all()
