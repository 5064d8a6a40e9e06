"""fp32 kernels on the fp32 matrix instruction (csrc/kernels/f32.hip) against fp64, at the borders of their rules and tiles."""
import pytest
import torch

from operator_amd import ops
from operator_amd.ops import decoder as dec

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _close(y, r, mag, K):
    """fp32 accumulation of K products: K 2^-24 of the sum of their magnitudes."""
    assert ((y.double() - r).abs() <= (K + 8) * 2.0 ** -24 * mag + 1e-30).all()


@pytest.mark.parametrize("M,N,K", [
    (1, 20, 16), (16, 64, 48), (17, 100, 2032), (17, 100, 2048), (32, 1000, 80), (33, 1000, 80), (64, 130, 512), (65, 68, 528),
    (130, 50, 16), (200, 2048, 1040), (257, 64, 4112)])
def test_gemm_f32_rules(M, N, K):
    torch.manual_seed(M + N + K)
    x, w = torch.randn(M, K, device=DEV), torch.randn(N, K, device=DEV)
    mag = x.double().abs() @ w.double().abs().t()
    _close(ops.linear_f32(x, w), x.double() @ w.double().t(), mag, K)
    gate, up = torch.randn(64, K, device=DEV) * K ** -0.5, torch.randn(64, K, device=DEV) * K ** -0.5
    y = ops.linear_f32(x, ops.interleave_gate_up(gate, up), ops.SILU).double()
    a, b = x.double() @ gate.double().t(), x.double() @ up.double().t()
    ma, mb = (x.double().abs() @ t.double().abs().t() for t in (gate, up))
    # silu's slope is below 1.1; expf and the quotient are within a few ulp
    err = (K + 8) * 2.0 ** -24 * (1.1 * ma * b.abs() + mb * a.abs()) + 2.0 ** -21 * (a * torch.sigmoid(a) * b).abs()
    assert ((y - a * torch.sigmoid(a) * b).abs() <= err + 1e-30).all()


@pytest.mark.parametrize("M", [1, 33, 70])
def test_head_gemm_f32(M):
    torch.manual_seed(M)
    x, w = torch.randn(M, 3, 88, device=DEV), torch.randn(3, 48, 80, device=DEV)
    y = torch.full((M, 3, 64), float("nan"), device=DEV)
    ops.kernels().head_gemm(x, w, y)
    r = torch.einsum("mhk,hnk->mhn", x[..., :80].double(), w.double())
    _close(y[..., :48], r, torch.einsum("mhk,hnk->mhn", x[..., :80].double().abs(), w.double().abs()), 80)
    assert y[..., 48:].isnan().all()


@pytest.mark.parametrize("M", [3, 33, 200])
@pytest.mark.parametrize("dx,dw", [(1, 0), (0, 2), (3, 3)])
def test_operands_off_their_alignment(M, dx, dw):
    """The tile kernel stages 16-B pieces; operands that start elsewhere give the same numbers."""
    torch.manual_seed(M + dx)

    def at(t, d):
        return torch.cat([torch.full((d,), float("nan"), device=DEV), t.flatten()])[d:].view(t.shape)

    x, w = torch.randn(M, 528, device=DEV), torch.randn(128, 528, device=DEV)
    xo, wo = at(x, dx), at(w, dw)
    assert (xo.data_ptr() % 16 == 0) == (dx == 0) and (wo.data_ptr() % 16 == 0) == (dw == 0)
    for glu in (0, ops.SILU):
        assert torch.equal(ops.linear_f32(xo, wo, glu), ops.linear_f32(x, w, glu))
    x, w = torch.randn(M, 2, 48, device=DEV), torch.randn(2, 32, 48, device=DEV)
    y, yo = (torch.empty(M, 2, 32, device=DEV) for _ in range(2))
    ops.kernels().head_gemm(x, w, y)
    ops.kernels().head_gemm(at(x, dx), at(w, dw), yo)
    assert torch.equal(y, yo)


def _attend(q, k, v, scale, window=0):
    n, T = k.shape[0], q.shape[0]
    s = torch.einsum("thd,jhd->htj", q.double(), k.double()) * scale
    i, j = torch.arange(n - T, n, device=DEV)[:, None], torch.arange(n, device=DEV)[None]
    hidden = (j > i) | ((i - j >= window) if window else False)
    return torch.einsum("htj,jhd->thd", torch.softmax(s.masked_fill(hidden, float("-inf")), -1), v.double())


@pytest.mark.parametrize("lens", [[1], [31, 32, 33], [64, 65, 200]])
@pytest.mark.parametrize("D,Dv,window", [(48, 32, 0), (128, 96, 40), (240, 256, 0)])
def test_prefill_attention_keeps_odd_values_to_their_queries(lens, D, Dv, window):
    """An infinity among the values of a token reaches the queries that see it and no other."""
    torch.manual_seed(len(lens) + D)
    H, G, T = 4, 2, sum(lens)
    L = dec.HeadLayout(H, G, D, Dv)
    q, k, v = (torch.randn(T, h, d, device=DEV) for h, d in ((H, D), (G, D), (G, Dv)))
    for odd in (False, True):
        bad = [sum(lens[:i]) + n - 1 - n // 3 for i, n in enumerate(lens)]
        if odd:
            v[bad, 0, 5] = float("inf")
        o = dec.attn_gd_prefill(q, k, v, lens, L, D ** -0.5, window=window).view(T, -1)[:, :H * Dv].view(T, H, Dv)
        a = 0
        for n, at in zip(lens, bad):
            clean = v[a:a + n].clone()
            clean[clean.isinf()] = 0.0
            r = _attend(q[a:a + n], k[a:a + n].repeat_interleave(H // G, 1), clean.repeat_interleave(H // G, 1), D ** -0.5, window)
            got = o[a:a + n]
            rows = torch.arange(a, a + n, device=DEV)
            sees = (rows >= at) & ((rows - at < window) if window else True)
            mask = torch.zeros_like(got, dtype=torch.bool)
            if odd:
                mask[:, :H // G, 5] = sees[:, None]
                assert (got[mask] == float("inf")).all()
            torch.testing.assert_close(got[~mask].double(), r[~mask], atol=2e-5, rtol=2e-5)
            a += n


@pytest.mark.parametrize("H,G,D,Dv,splits,window", [(40, 2, 64, 64, 1, 0), (4, 4, 128, 160, 3, 0), (16, 1, 256, 256, 4, 0), (6, 2, 48, 32, 2, 50)])
def test_decode_attention_pieces(H, G, D, Dv, splits, window):
    torch.manual_seed(H + D)
    P, ctx = 16, [1, 0, 15, 16, 17, 130, 500]
    L, B = dec.HeadLayout(H, G, D, Dv), len(ctx)
    pages = [-(-n // P) for n in ctx]
    perm = torch.randperm(sum(pages) + 1).int()
    kc, vc = (torch.full((len(perm), G, P, d), float("nan"), device=DEV) for d in (D, Dv))   # what no token wrote stays out
    bt = torch.zeros(B, max(pages), dtype=torch.int32)
    q, seqs, at = torch.randn(B, H, D, device=DEV), [], 0
    for b, n in enumerate(ctx):
        bt[b, :pages[b]] = perm[at:at + pages[b]]
        at += pages[b]
        k, v = torch.randn(n, G, D, device=DEV), torch.randn(n, G, Dv, device=DEV)
        for t in range(n):
            kc[bt[b, t // P], :, t % P], vc[bt[b, t // P], :, t % P] = k[t], v[t]
        seqs.append((k, v))
    gate = torch.rand(B, H, device=DEV)
    o = dec.attn_gd_decode(q, (kc, vc), bt.to(DEV), torch.tensor(ctx, dtype=torch.int32, device=DEV), L, D ** -0.5, splits, window=window,
                           gate=gate)[:, :H * Dv].view(B, H, Dv)
    for b, (k, v) in enumerate(seqs):
        if ctx[b] == 0:
            assert (o[b] == 0).all()
            continue
        r = _attend(q[b:b + 1], k.repeat_interleave(H // G, 1), v.repeat_interleave(H // G, 1), D ** -0.5, window)[0]
        torch.testing.assert_close(o[b].double(), r * gate[b].double()[:, None], atol=2e-5, rtol=2e-5)


@pytest.mark.parametrize("D,Dv", [(4, 1), (20, 18), (36, 100), (132, 130), (256, 255), (20, 96), (64, 17)])
def test_prefill_attention_unpadded_heads(D, Dv):
    """Key heads of any multiple of 4 columns, value heads of any number; columns past the heads stay as they are."""
    torch.manual_seed(D + Dv)
    H, G, lens = 4, 2, [1, 70, 131]
    T = sum(lens)
    L = dec.HeadLayout(H, G, D, Dv)
    q, k, v = (torch.randn(T, h, d, device=DEV) for h, d in ((H, D), (G, D), (G, Dv)))
    o = dec.attn_gd_prefill(q, k, v, lens, L, D ** -0.5, window=50)
    a = 0
    for n in lens:
        r = _attend(q[a:a + n], k[a:a + n].repeat_interleave(H // G, 1), v[a:a + n].repeat_interleave(H // G, 1), D ** -0.5, 50)
        torch.testing.assert_close(o[a:a + n, :H * Dv].view(n, H, Dv).double(), r, atol=2e-5, rtol=2e-5)
        a += n
    assert (o[:, H * L.pads[1]:] == 0).all()


@pytest.mark.parametrize("D,Dv", [(4, 1), (20, 18), (36, 100), (132, 130), (640, 639), (20, 320), (64, 17)])
@pytest.mark.parametrize("splits", [1, 3])
def test_decode_attention_unpadded_heads(D, Dv, splits):
    torch.manual_seed(D + Dv)
    P, ctx, H, G = 16, [1, 0, 17, 200], 6, 2
    L, B, pages = dec.HeadLayout(H, G, D, Dv), len(ctx), 13
    kc, vc = (torch.full((B * pages, G, P, d), float("nan"), device=DEV) for d in (D, Dv))
    bt = torch.arange(B * pages, dtype=torch.int32).flip(0).view(B, pages).contiguous()   # the last page is read to its end
    q = torch.randn(B, H, D, device=DEV)
    seqs = []
    for b, n in enumerate(ctx):
        k, v = torch.randn(n, G, D, device=DEV), torch.randn(n, G, Dv, device=DEV)
        for t in range(n):
            kc[bt[b, t // P], :, t % P], vc[bt[b, t // P], :, t % P] = k[t], v[t]
        seqs.append((k, v))
    o = dec.attn_gd_decode(q, (kc, vc), bt.to(DEV), torch.tensor(ctx, dtype=torch.int32, device=DEV), L, D ** -0.5, splits)
    for b, (k, v) in enumerate(seqs):
        got = o[b, :H * Dv].view(H, Dv)
        if ctx[b] == 0:
            assert (got == 0).all()
            continue
        r = _attend(q[b:b + 1], k.repeat_interleave(H // G, 1), v.repeat_interleave(H // G, 1), D ** -0.5)[0]
        torch.testing.assert_close(got.double(), r, atol=2e-5, rtol=2e-5)


@pytest.mark.parametrize("rank,splits", [(256, 2), (544, 1), (608, 3)])
def test_latent_decode_f32_wide_rows(rank, splits):
    torch.manual_seed(rank)
    P, ctx, H, rot = 16, [3, 40, 200], 18, 32
    L = dec.LatentLayout(H, 64, rot, 64, 128, rank)
    B, pages = len(ctx), 1 + max(-(-n // P) for n in ctx)
    cache = torch.full((B * pages, 1, P, L.ck), float("nan"), device=DEV)
    bt = torch.arange(B * pages, dtype=torch.int32).view(B, pages)
    rows = [torch.randn(n, L.ck, device=DEV) for n in ctx]
    for b, r in enumerate(rows):
        r[:, L.rp + rot:] = 0
        cache[b * pages:(b + 1) * pages].view(-1, L.ck)[:ctx[b]] = r
    q = torch.randn(B, H, L.ck, device=DEV)
    o = dec.attn_latent_decode(q, cache, bt.to(DEV), torch.tensor(ctx, dtype=torch.int32, device=DEV), L, 0.05, splits)
    for b, r in enumerate(rows):
        p = torch.softmax(q[b].double() @ r.double().t() * 0.05, -1)
        torch.testing.assert_close(o[b].double(), p @ r.double()[:, :L.rp], atol=2e-5, rtol=2e-5)


@pytest.mark.parametrize("M,N,K,S", [(1, 4, 16, 1), (33, 100, 48, 1), (64, 130, 528, 1), (65, 128, 2032, 3), (129, 260, 1040, 2), (257, 1000, 96, 3),
                                     (300, 128, 4112, 8), (40, 64, 16, 2)])
def test_gemm_f32_split(M, N, K, S):
    """Ragged tiles, a last piece of 16 columns, slices (empty ones too): the bits do not depend on the tile's rows, and the sums are no
    further from the 64-bit result than the fp32 instruction's."""
    torch.manual_seed(M + N + K)
    x, w = torch.randn(M, K, device=DEV), torch.randn(N, K, device=DEV)
    C, r, mag = ops.kernels(), x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()

    def run(rows, splits, w=w, n=N, glu=0):
        y = torch.full((M, n), float("nan"), device=DEV)
        part = torch.full((splits * M * w.shape[0],), float("nan"), device=DEV) if splits > 1 else None
        C.gemm_f32(x, w, y, glu, partial=part, splits=splits, rows=rows)
        return y

    for s in {1, S if N % 4 == 0 else 1}:
        ys = [run(rows, s) for rows in (64, 128, 256)]
        assert torch.equal(ys[0], ys[1]) and torch.equal(ys[0], ys[2])
        _close(ys[0], r, mag, K)
        if K >= 512:
            assert (ys[0].double() - r).norm() <= 1.02 * (run(0, 1).double() - r).norm()
    gate, up = torch.randn(128, K, device=DEV) * K ** -0.5, torch.randn(128, K, device=DEV) * K ** -0.5
    wgu = ops.interleave_gate_up(gate, up)
    a, b = x.double() @ gate.double().t(), x.double() @ up.double().t()
    for s in {1, S}:
        ys = [run(rows, s, wgu, 128, ops.SILU) for rows in (64, 128, 256)]
        assert torch.equal(ys[0], ys[1]) and torch.equal(ys[0], ys[2])
        torch.testing.assert_close(ys[0].double(), a * torch.sigmoid(a) * b, atol=2e-5, rtol=2e-5)


@pytest.mark.parametrize("rows,S", [(64, 1), (128, 2), (256, 1)])
def test_gemm_f32_split_keeps_odd_values_and_small_ones(rows, S):
    """Infinities, NaN and operands whose parts leave bf16's range give what 32-bit products give, in their own rows and columns."""
    torch.manual_seed(rows)
    M, N, K = 300, 260, 96
    x, w = torch.randn(M, K, device=DEV), torch.randn(N, K, device=DEV)
    x[3, 5], x[200, 95], x[77, 0], w[131, 7] = float("inf"), float("-inf"), float("nan"), float("inf")
    x[150] *= 1e-36           # third parts below bf16's range
    w[40:45] *= 1e-30
    x[20, 9], w[200, 3] = 3.4e38, -3.4028234e38   # round to an infinity in bf16
    x[30] = 0
    y = torch.empty(M, N, device=DEV)
    part = torch.empty(S * M * N, device=DEV) if S > 1 else None
    ops.kernels().gemm_f32(x, w, y, 0, partial=part, splits=S, rows=rows)
    r = (x.double() @ w.double().t())
    r32, mag = r.float(), x.double().abs() @ w.double().abs().t()
    assert torch.equal(y.isnan(), r32.isnan()) and torch.equal(y.isinf() & ~r.isinf(), r32.isinf() & ~r.isinf())
    assert torch.equal(y[r.isinf()], r32[r.isinf()])
    fin = r.isfinite() & r32.isfinite()
    assert ((y[fin].double() - r[fin]).abs() <= (K + 8) * 2.0 ** -24 * mag[fin] + 1e-44).all()


def _split(x, w, rows, S=1, glu=0):
    M, N = x.shape[0], w.shape[0]
    y = torch.full((M, N // 2 if glu else N), float("nan"), device=DEV)
    part = torch.full((S * M * N,), float("nan"), device=DEV) if S > 1 else None
    ops.kernels().gemm_f32(x, w, y, glu, partial=part, splits=S, rows=rows)
    return y


@pytest.mark.parametrize("S", [1, 3])
@pytest.mark.parametrize("glu", [0, ops.SILU])
def test_gemm_f32_split_odd_values_leave_other_rows_as_they_are(S, glu):
    """What is done again in 32-bit products is the odd sum alone: other rows and columns keep their bits, and so do all between tile rows."""
    torch.manual_seed(S)
    M, N, K = 300, 256, 112
    x, w = torch.randn(M, K, device=DEV), torch.randn(N, K, device=DEV)
    before = [_split(x, w, rows, S, glu) for rows in (64, 128, 256)]
    x[3, 5], x[77, 0], w[131, 7] = float("inf"), float("nan"), float("-inf")
    x[150] *= 1e-36
    w[40] *= 1e-30
    after = [_split(x, w, rows, S, glu) for rows in (64, 128, 256)]
    r, c = torch.ones(M, dtype=torch.bool, device=DEV), torch.ones(N, dtype=torch.bool, device=DEV)
    r[[3, 77, 150]] = False
    c[[131, 40]] = False
    if glu:   # a feature's gate and up
        c = c.view(-1, 2, 64).all(1).flatten()
    for y, z in zip(before, after):
        assert torch.equal(y[r][:, c], z[r][:, c])
        assert ((z == after[0]) | (z.isnan() & after[0].isnan())).all()


@pytest.mark.parametrize("rows,S", [(64, 1), (128, 3), (256, 1)])
@pytest.mark.parametrize("small,large", [(1e-36, 1e20), (1e-38, 1e22), (1e-41, 1e30), (1e-41, 1e9), (1e-30, 2e9), (1e-15, 1.0)])
def test_gemm_f32_split_small_operands_beside_large_ones(small, large, rows, S):
    """Operands whose parts leave bf16's range count where their partners are large: sums of them are what 32-bit products give, whether a row is
    small all along or in one place, also where every part of it rounds to zero."""
    torch.manual_seed(rows)
    M, N, K = 150, 260, 272
    x, w = torch.randn(M, K, dtype=torch.float64), torch.randn(N, K, dtype=torch.float64)
    x[:40] *= small
    w[:192] *= large   # whole blocks of sums without a small one
    x[60:70] = 0.0
    x[60:65, 100] = small
    w[192:230] *= small
    x[100:120, 3::4] *= large
    x, w = x.float().to(DEV), w.float().to(DEV)
    y, r = _split(x, w, rows, S), x.double() @ w.double().t()
    mag = x.double().abs() @ w.double().abs().t()
    fin = mag < 1e38
    assert ((y.double() - r).abs() <= (K + 8) * 2.0 ** -24 * mag + K * 2.0 ** -149)[fin].all()
    plain = _split(x, w, 0)   # the fp32 instruction: as close, but for the order of the sums
    for a, b in ((slice(0, 40), slice(0, 192)), (slice(100, 120), slice(192, 230))):
        err, ref = ((t.double() - r)[a, b].norm() for t in (y, plain))
        assert err <= 1.25 * ref


@pytest.mark.parametrize("rows", [64, 256])
def test_gemm_f32_split_drops_no_more_than_a_rounding(rows):
    """Operands of which the products left out add up to the most: 2^-24 of each product, all to one side."""
    x, w = (torch.full((n, 16), 1.0038986, device=DEV) for n in (70, 130))
    r = x.double() @ w.double().t()
    assert ((_split(x, w, rows).double() - r).abs() <= (1 + 6) * 2.0 ** -24 * r).all()   # and six roundings of the sum
