"""gemm_decode and the experts' tiles start their K steps by column tile and expert: fewer steps than tiles, one step, uneven slices, tiled
weights, against float64."""
import pytest
import torch

from operator_amd import ops
from operator_amd.ops import decoder, reference

pytestmark = pytest.mark.gpu


# fp32 sums of K products of bf16 numbers (exact each), then one rounding to bf16
def _check(y, x, w, K):
    want, mag = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    assert ((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + (K + 16) * 2.0 ** -24 * mag).all()


# on either side of the columns and the X (2^20) that turn and of 2048 columns apart, 128-row tiles over 64 columns, which never do
@pytest.mark.parametrize("M,N,K,S,bn,bm,stages", [
    (64, 1152, 192, 3, 64, 64, 3), (64, 524288, 64, 1, 128, 64, 3), (64, 175360, 192, 3, 64, 64, 3), (64, 32768, 1024, 1, 128, 64, 4),
    (64, 25024, 1344, 5, 64, 64, 6), (128, 75008, 448, 2, 128, 64, 2), (128, 4096, 8192, 1, 128, 128, 4), (128, 4096, 8256, 3, 128, 128, 3),
    (128, 32768, 1024, 1, 64, 128, 4), (256, 32768, 1024, 1, 128, 256, 3)])
def test_steps_go_round(M, N, K, S, bn, bm, stages):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x, w = (torch.randn(n, K, generator=g, device="cuda").bfloat16() for n in (M, N))
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    p = torch.full((S, M, N), float("nan"), device="cuda") if S > 1 else None
    C = ops.kernels()
    C.gemm_decode(x, w, y, p, S, bn, bm, False, False, stages)
    _check(y, x, w, K)
    wt = w.view(N // 64, 64, K // 64, 64).transpose(1, 2).contiguous().view(N, K)
    C.gemm_decode(x, wt, y.fill_(float("nan")), p, S, bn, bm, False, True, stages)
    _check(y, x, w, K)


@pytest.mark.parametrize("T,E,ld,ff,top,plan", [(9, 7, 128, 128, 2, 64), (70, 3, 256, 192, 1, 64), (40, 16, 384, 64, 4, 128), (17, 8, 2048, 1024, 2, None)])
def test_experts(T, E, ld, ff, top, plan):
    g = torch.Generator(device="cuda").manual_seed(T + E)
    h = torch.randn(T, ld, generator=g, device="cuda").bfloat16()
    ids = torch.rand(T, E, generator=g, device="cuda").topk(top).indices.int()
    wt = torch.rand(T, top, generator=g, device="cuda")
    wgu = (torch.randn(E, 2 * ff, ld, generator=g, device="cuda") * ld ** -0.5).bfloat16()
    wd = (torch.randn(E, ld, ff, generator=g, device="cuda") * ff ** -0.5).bfloat16()
    y, pos = decoder.experts(h, ids, wt, wgu, wd, plan)
    got = y[pos.long()] if pos is not None else y.view(T, top, ld)
    want = reference.experts(h.cpu().float(), ids.cpu(), wt.cpu(), wgu.cpu().float(), wd.cpu().float()).view(T, top, ld).to("cuda")
    # the gated product is rounded to bf16 (2^-8 of each, a random sum over ff: against the size of a row), the result once more
    assert ((got.float() - want).abs() <= 6 * 2.0 ** -9 * want.norm(dim=-1, keepdim=True) + 2.0 ** -8 * want.abs()).all()


@pytest.mark.parametrize("M,N,K,ns", [(64, 32768, 1024, 4), (64, 33024, 1088, 3), (128, 32768, 1088, 4), (128, 32768, 1088, 3), (128, 1024, 1088, 4)])
def test_gated(M, N, K, ns):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    y = torch.full((M, N // 2), float("nan"), dtype=torch.bfloat16, device="cuda")
    ops.kernels().gemm_decode(x, w, y, None, 1, 128, M, 1, False, ns)
    r = (x.double() @ w.double().t()).view(M, N // 128, 2, 64)
    gate, up = r[:, :, 0].reshape(M, -1), r[:, :, 1].reshape(M, -1)
    sg = torch.nn.functional.silu(gate)
    # gate, silu(gate), up and the product are rounded to bf16: 2^-8 of each (silu's slope is at most 1.1); second order and the fp32 sums
    tol = 1.02 * 2.0 ** -8 * up.abs() * (1.1 * gate.abs() + 3 * sg.abs()) + 1e-4 * (1 + up.abs() + gate.abs())
    assert ((y.double() - sg * up).abs() <= tol).all()


@pytest.mark.parametrize("M,N,K,bn,bm,turn", [
    (64, 16384, 2048, 128, 64, True), (64, 16256, 2048, 128, 64, False), (64, 16384, 4096, 64, 64, True), (64, 28672, 3584, 128, 64, False),
    (64, 34176, 4160, 128, 64, False), (128, 24576, 2048, 64, 64, True), (128, 24512, 2048, 64, 64, False), (128, 32768, 4096, 128, 128, True),
    (128, 28672, 4096, 128, 128, False), (128, 34176, 4032, 128, 128, False)])
def test_only_rows_a_multiple_of_2048_columns_apart_turn(M, N, K, bn, bm, turn):
    """Where steps go round a column's sum depends on its tile, elsewhere it does not."""
    g = torch.Generator(device="cuda").manual_seed(N + K)
    x, w = (torch.randn(n, K, generator=g, device="cuda").bfloat16() for n in (M, N))
    C, at = ops.kernels(), bn * 37
    y, z = (torch.empty(M, n, device="cuda").bfloat16() for n in (N, bn))
    C.gemm_decode(x, w, y, None, 1, bn, bm, False, False, 3)
    C.gemm_decode(x, w[at:at + bn].contiguous(), z, None, 1, bn, bm, False, False, 3)   # one tile: in step
    assert torch.equal(y[:, at:at + bn], z) != turn
