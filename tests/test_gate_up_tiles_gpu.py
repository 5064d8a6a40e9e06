"""Gated decode tiles of 64 and 160 columns: the bits of the 128-column ones where the K steps have the same order, fp64 elsewhere; features that do
not fill the last tile, K shorter than the ring, both activations; and the rule that chooses them."""
import pytest
import torch

from operator_amd import ops
from operator_amd.ops import reference as ref

DEV = "cuda"


def _rand(*shape, scale=1.0):
    return (torch.randn(*shape, device=DEV) * scale).to(torch.bfloat16)


# one tile, features that end inside a tile of 160 or of 64, several rounds; one K step, fewer than the ring's, odd numbers of them; K whose steps go
# round (16384 x 2048, 37888 x 2048)
@pytest.mark.gpu
@pytest.mark.parametrize("inter,K", [(64, 64), (128, 192), (192, 320), (8192, 448), (20544, 128), (8192, 2048), (18944, 2048)])
@pytest.mark.parametrize("act", [ops.SILU, ops.GELU_TANH])
def test_gated_tiles(inter, K, act):
    torch.manual_seed(inter + K)
    C, g, u = ops.kernels(), _rand(inter, K, scale=0.05), _rand(inter, K, scale=0.05)
    w, x = ops.interleave_gate_up(g, u), _rand(256, K)
    gate, up = ((x.double() @ t.double().t()).to(torch.bfloat16) for t in (g, u))
    r = ref.silu_mul(torch.cat([gate, up], 1), None, act == ops.GELU_TANH).double()
    # each of gate, act(gate) and up may round the other way (2^-8; the activation's slope is below 1.2), and a gate or an up near 0 carries the absolute
    # error of its fp32 sum, K 2^-24 of the sum of magnitudes
    sum_g, sum_u = (K * 2.0 ** -24 * (x.double().abs() @ t.double().abs().t()) for t in (g, u))
    bound = 5 * 2.0 ** -8 * r.abs() + 1.2 * up.double().abs() * (2.0 ** -8 * gate.double().abs() + sum_g) + gate.double().abs() * sum_u + 1e-6
    for M in (64, 128, 256):
        for (bm, bn), ns in ops._GU_TILES.items():
            if M % bm:
                continue
            guard = torch.full((M + 1, inter), float("nan"), dtype=torch.bfloat16, device=DEV)
            y, want = guard[:M], torch.empty(M, inter, dtype=torch.bfloat16, device=DEV)
            C.gemm_decode(x[:M], w, y, None, 1, bn, bm, act, False, ns)
            assert guard[M:].isnan().all() and ((y.double() - r[:M]).abs() <= bound[:M]).all(), (M, bm, bn)
            if K % 2048 or bn == 64:
                C.gemm_decode(x[:M], w, want, None, 1, 128, bm, act, False, 3)
                assert torch.equal(y, want), (M, bm, bn)


@pytest.mark.gpu
def test_other_widths_are_refused():
    x, w, y = _rand(64, 128), _rand(512, 128), torch.empty(64, 256, dtype=torch.bfloat16, device=DEV)
    for bn, act, tiled in ((96, 1, False), (192, 1, False), (64, 1, True), (160, 0, False)):
        with pytest.raises(RuntimeError):
            ops.kernels().gemm_decode(x, w, y if act else torch.empty(64, 512, dtype=torch.bfloat16, device=DEV), None, 1, bn, 64, act, tiled, 3)


def test_the_width_that_is_one_round():
    assert [ops.gate_up_tile(M, 37888, 3584) for M in (64, 128, 256)] == [(64, 160, 4), (128, 160, 3), (256, 160, 3)]
    assert ops.gate_up_tile(64, 16384, 2048) == (64, 64, 4) and ops.gate_up_tile(256, 8192, 4096) == (128, 64, 4)
    # as fast or faster in tiles of 128 columns, or cut along K
    for M, N, K in ((64, 28672, 4096), (128, 28672, 4096), (256, 28672, 4096), (128, 16384, 2048), (64, 57344, 8192), (64, 8192, 4096), (64, 4096, 2048),
                    (192, 12288, 2048), (192, 37888, 3584)):
        assert ops.gate_up_tile(M, N, K) is None, (M, N, K)
    for M in (64, 128, 192, 256):
        for N in range(128, 65536, 896):
            t = ops.gate_up_tile(M, N - N % 128, 2048)
            assert t is None or (M % t[0] == 0 and t == (*t[:2], ops._GU_TILES[t[:2]]) and 96 <= M // t[0] * -(-(N - N % 128) // t[1]) <= ops.CUS)
