"""Prefill attention at the edges of its 64-key tiles and 32-row blocks: every group size, what lies behind a sequence's last key,
and scales that are not positive (the running maximum is taken before the scale), against 64 bits."""
import pytest
import torch

from operator_amd import ops
from operator_amd.ops import decoder as dec

DEV = "cuda"


def _exact(q, k, v, lens, scale, window=1 << 30):
    out, a, per = [], 0, q.shape[1] // k.shape[1]
    for n in lens:
        i = torch.arange(n, device=DEV)
        hidden = (i[None, :] > i[:, None]) | (i[:, None] - i[None, :] >= window)
        for h in range(q.shape[1]):
            s = (q[a:a + n, h].double() @ k[a:a + n, h // per].double().t()) * scale
            out.append(torch.softmax(s.masked_fill(hidden, -torch.inf), -1) @ v[a:a + n, h // per].double())
        a += n
    o, r = [], 0
    for n in lens:
        o.append(torch.stack(out[r:r + q.shape[1]], 1))
        r += q.shape[1]
    return torch.cat(o)


def _close(o, r, v):
    # the weights are rounded to bf16 before the values (2^-8 of each, at most that of the largest value in all) and the result once
    assert ((o.double() - r).abs() <= 2.0 ** -8 * (r.abs() + v.double().abs().max()) + 1e-6).all()


LENS = [1, 31, 33, 63, 64, 65, 127, 129, 200]


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv", [(2, 2), (4, 2), (3, 1), (8, 2), (5, 1), (7, 1), (8, 1)])
@pytest.mark.parametrize("scale", [128 ** -0.5, -0.07, 0.0])
def test_rows_and_scales(Hq, Hkv, scale):
    torch.manual_seed(Hq)
    T = sum(LENS)
    # the rows behind the last sequence are NaN: a tile's rows past the end are never multiplied
    buf = [torch.full((T + 64, h, 128), float("nan"), dtype=torch.bfloat16, device=DEV) for h in (Hkv, Hkv)]
    for b in buf:
        b[:T] = torch.randn(T, Hkv, 128, device=DEV).bfloat16()
    q, (k, v) = torch.randn(T, Hq, 128, device=DEV).bfloat16(), (b[:T] for b in buf)
    _close(ops.attn_prefill(q, k, v, LENS, scale), _exact(q, k, v, LENS, scale), v)


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [0.11, -0.07, 0.0])
@pytest.mark.parametrize("window", [50, 64, 0])
def test_windows_and_scales(scale, window):
    torch.manual_seed(window)
    T, Hq, Hkv, dk, dv = sum(LENS), 4, 2, 96, 64   # sizes that need no padding
    L = dec.HeadLayout(Hq, Hkv, dk, dv)
    assert L.pads == (dk, dv) and L.ocol == Hq * dv
    q, k, v = (torch.randn(T, h, d, device=DEV).bfloat16() for h, d in ((Hq, dk), (Hkv, dk), (Hkv, dv)))
    o = dec.attn_gd_prefill(q, k, v, LENS, L, scale, window=window)
    _close(o.view(T, Hq, dv), _exact(q, k, v, LENS, scale, window or 1 << 30), v)


def _off(t, shift):
    """t's rows ``shift`` elements past a 16-byte alignment."""
    b = torch.empty(t.numel() + shift, dtype=t.dtype, device=DEV)[shift:].view(t.shape)
    return b.copy_(t)


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv", [(4, 2), (7, 1)])
@pytest.mark.parametrize("shift", [1, 2, 4])
def test_keys_off_their_alignment(Hq, Hkv, shift):
    """Keys and values off 16 bytes, own and of a prefix, come as a copy: the same bits."""
    torch.manual_seed(shift)
    lens, P = [70, 33, 130], 100
    T = sum(lens)
    q, k, v = (torch.randn(T, h, 128, device=DEV).bfloat16() for h in (Hq, Hkv, Hkv))
    pk, pv = (torch.randn(P, Hkv, 128, device=DEV).bfloat16() for _ in range(2))
    var = ops.prefill_variant(Hq, Hkv)
    ws, wq = ops.prefill_work_list(lens, ops.prefill_block_q(Hq, Hkv, var))
    work = tuple(torch.tensor(t, dtype=torch.int32, device=DEV) for t in ([0, 70, 103, 233], ws, wq)) + (var,)
    sp = torch.full((3,), P, dtype=torch.int32, device=DEV)
    assert _off(k, shift).data_ptr() % 16 == 2 * shift
    for pre, pre_off in ((None, None), ((pk, pv, sp, [P] * 3), (_off(pk, shift), _off(pv, shift), sp, [P] * 3))):
        want = ops.attn_prefill(q, k, v, lens, 0.09, work=work, prefix=pre)
        assert torch.equal(ops.attn_prefill(q, _off(k, shift), _off(v, shift), lens, 0.09, work=work, prefix=pre_off), want)


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv", [(4, 2), (8, 1)])
@pytest.mark.parametrize("P", [1, 63, 65, 100])
def test_prefix_ends_inside_a_tile(Hq, Hkv, P):
    """What stands behind the last row of a prefix is NaN, and so is what stands behind the own rows: neither is ever multiplied."""
    torch.manual_seed(P)
    lens = [1, 40, 65]
    T, nan = sum(lens), float("nan")
    q = torch.randn(T, Hq, 128, device=DEV).bfloat16()
    pk, pv, k, v = (torch.full((n + 64, Hkv, 128), nan, dtype=torch.bfloat16, device=DEV) for n in (P, P, T, T))
    for t, n in ((pk, P), (pv, P), (k, T), (v, T)):
        t[:n] = torch.randn(n, Hkv, 128, device=DEV).bfloat16()
    var = ops.prefill_variant(Hq, Hkv)
    ws, wq = ops.prefill_work_list(lens, ops.prefill_block_q(Hq, Hkv, var))
    work = tuple(torch.tensor(t, dtype=torch.int32, device=DEV) for t in ([0, 1, 41, 106], ws, wq)) + (var,)
    sp = torch.full((3,), P, dtype=torch.int32, device=DEV)
    o, a = ops.attn_prefill(q, k[:T], v[:T], lens, 128 ** -0.5, work=work, prefix=(pk, pv, sp, [P] * 3)), 0
    for n in lens:
        kk, vv = torch.cat([pk[:P], k[a:a + n]]), torch.cat([pv[:P], v[a:a + n]])
        qq = torch.cat([torch.zeros(P, Hq, 128, dtype=q.dtype, device=DEV), q[a:a + n]])   # rows of their own for the prefix, not looked at
        _close(o[a:a + n], _exact(qq, kk, vv, [P + n], 128 ** -0.5)[P:], vv)
        a += n
