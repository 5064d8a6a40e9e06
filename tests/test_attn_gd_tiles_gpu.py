"""Prefill attention of general head sizes, key and value tiles brought by LDS-DMA: every instantiated pair of sizes and sizes between them, NaN rows
behind the last sequence, keys and values off 16 bytes, and what is left of a prefix tile, against 64 bits."""
import pytest
import torch

from operator_amd.ops import decoder as dec

DEV = "cuda"
LENS = [1, 63, 65, 130]


def _exact(q, k, v, lens, scale, pk, pv, window):
    o, a, per, P = [], 0, q.shape[1] // k.shape[1], pk.shape[0]
    for n in lens:
        kk, vv = (torch.cat([p, t[a:a + n]]).double().repeat_interleave(per, 1) for p, t in ((pk, k), (pv, v)))
        at = torch.arange(P + n, device=DEV)
        back = at[P:, None] - at[None]
        s = torch.einsum("qhd,khd->hqk", q[a:a + n].double(), kk) * scale
        w = torch.softmax(s.masked_fill((back < 0) | (back >= window), -torch.inf), -1)
        o.append(torch.einsum("hqk,khd->qhd", w, vv))
        a += n
    return torch.cat(o)


def _close(o, r, v):
    # the weights are rounded to bf16 before the values (2^-8 of each, at most that of the largest value in all) and the result once
    assert ((o.double() - r).abs() <= 2.0 ** -8 * (r.abs() + v.double().abs().max()) + 1e-6).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dk", [24, 32, 64, 80, 96, 128, 160, 192, 224, 256])
@pytest.mark.parametrize("dv", [32, 64, 96, 128, 160, 256])
@pytest.mark.parametrize("H,G", [(4, 1), (2, 2)])
def test_head_sizes(dk, dv, H, G):
    torch.manual_seed(dk + dv)
    T, P = sum(LENS), 70
    q = torch.randn(T, H, dk, device=DEV).bfloat16()
    k, v, pk, pv = (torch.full((n + 64, G, d), float("nan"), dtype=torch.bfloat16, device=DEV) for n, d in ((T, dk), (T, dv), (P, dk), (P, dv)))
    for t, n in ((k, T), (v, T), (pk, P), (pv, P)):
        t[:n] = torch.randn(n, G, t.shape[2], device=DEV).bfloat16()
    k, v, pk, pv = k[:T], v[:T], pk[:P], pv[:P]
    C, i32 = dec.kernels(), lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)   # noqa: E731
    cu = i32([0] + [sum(LENS[:i + 1]) for i in range(len(LENS))])
    items = [(s, r) for s, n in enumerate(LENS) for r in range(0, n, 128)]
    ws, wq = i32([s for s, _ in items]), i32([r for _, r in items])

    def run(k, v, pk, pv, pfx, window):
        o = torch.full((T, H * dv), float("nan"), dtype=torch.bfloat16, device=DEV)
        C.attn_gd_prefill(q, k, v, o, cu, ws, wq, dk ** -0.5, pk, pv, pfx, window, None)
        return o.view(T, H, dv)

    none = k[:0], v[:0]
    _close(run(k, v, None, None, None, 0), _exact(q, k, v, LENS, dk ** -0.5, *none, 1 << 30), v)
    _close(run(k, v, None, None, None, 50), _exact(q, k, v, LENS, dk ** -0.5, *none, 50), v)
    pfx = i32([P] * len(LENS))
    o = run(k, v, pk, pv, pfx, 0)
    _close(o, _exact(q, k, v, LENS, dk ** -0.5, pk, pv, 1 << 30), torch.cat([v, pv]))

    def off(t):
        return torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)[1:].view(t.shape).copy_(t)

    assert torch.equal(run(off(k), off(v), off(pk), off(pv), pfx, 0), o)
