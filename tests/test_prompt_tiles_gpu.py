"""gemm_mid's tiles of 64 to 256 rows and 64, 128 or 256 columns sum in the same order as its 128 x 256 ones: the same bits for every epilogue, at
edges of tiles and remainders, with K shorter than the ring and several rounds of tiles per workgroup; and the rule that chooses them."""
import pytest
import torch

from operator_amd import ops

DEV = "cuda"
TILES = [(64, 64), (128, 64), (64, 128), (96, 128), (128, 128), (160, 128), (192, 128), (224, 128), (256, 128), (64, 256)]


def _rand(*shape, scale=1.0):
    return (torch.randn(*shape, device=DEV) * scale).to(torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,S", [(1, 16, 64, 1), (63, 128, 128, 2), (64, 272, 192, 3), (65, 528, 320, 1), (100, 384, 448, 2), (129, 256, 1024, 5),
                                     (161, 1040, 128, 1), (225, 144, 128, 2), (257, 4112, 256, 1), (320, 6144, 64, 1), (700, 16400, 192, 1), (130, 8192, 576, 4)])
def test_every_tile_gives_the_same_bits(M, N, K, S):
    torch.manual_seed(M + N + K)
    C, x, w, b = ops.kernels(), _rand(M, K), _rand(N, K, scale=0.05), _rand(N)
    new = lambda *s, dt=torch.bfloat16: torch.full(s, float("nan"), dtype=dt, device=DEV)  # noqa: E731
    if S > 1:
        C.gemm_mid(x, w, None, b, want := new(S, M, N, dt=torch.float32), S)
    for rows, cols in TILES:
        opt = dict(rows=rows, cols=cols)
        if S > 1:
            C.gemm_mid(x, w, None, b, p := new(S, M, N, dt=torch.float32), S, **opt)
            assert torch.equal(p, want), opt
            continue
        for bias in (None, b):
            C.gemm_mid(x, w, y0 := new(M, N), bias)
            wide = new(M, N + 64)
            C.gemm_mid(x, w, wide[:, 32:32 + N], bias, **opt)
            assert torch.equal(wide[:, 32:32 + N], y0) and wide[:, :32].isnan().all() and wide[:, 32 + N:].isnan().all(), opt
    if N % 128 == 0:
        for act in (ops.SILU, ops.GELU_TANH):
            C.gemm_mid(x, w, y0 := new(M, N // 2), None, new(S, M, N, dt=torch.float32), S, act)
            for rows, cols in TILES:
                if cols > 64 or S > 1:
                    C.gemm_mid(x, w, y := new(M, N // 2), None, new(S, M, N, dt=torch.float32), S, act, rows=rows, cols=cols)
                    assert torch.equal(y, y0), (rows, cols, act)


@pytest.mark.gpu
@pytest.mark.parametrize("opt", [dict(rows=96, cols=64), dict(rows=160, cols=64), dict(rows=192, cols=64), dict(rows=224, cols=256), dict(rows=64, cols=192), dict(rows=32, cols=128), dict(rows=64, cols=64, silu_gu=1)])
def test_other_tiles_are_refused(opt):
    x, w = _rand(40, 128), _rand(256, 128)
    with pytest.raises(RuntimeError):
        ops.kernels().gemm_mid(x, w, torch.empty(40, 128 if "silu_gu" in opt else 256, dtype=torch.bfloat16, device=DEV), **opt)


def test_tiles_that_the_kernels_have():
    for N, K in ((16, 128), (272, 192), (4096, 4096), (28672, 4096), (3584, 18944), (37888, 3584)):
        for M in (1, 24, 33, 64, 65, 128, 129, 300, 885, 2048, 2049, 4096, 4097, 30000):
            for S in (1, 2, 8):
                for glu in (0, ops.SILU):
                    t = ops.prompt_tile(M, N, K, S, glu)
                    assert t in TILES or t == (ops.tile_rows(M, N, K, S), 256)
                    assert t[1] > 64 or S > 1 or not glu
    # both sides timed (us): 18 and 31, 29 and 55, 56 and 65; 49 and 45, 101 and 96; 47 and 40
    assert [ops.prompt_tile(100, *a) for a in ((6144, 4096, 2), (4096, 14336, 4), (28672, 4096, 1, 1))] == [(128, 64), (128, 64), (128, 128)]
    assert [ops.prompt_tile(885, *a) for a in ((6144, 4096, 1), (4096, 14336, 2))] == [(192, 128), (224, 128)]
    assert ops.prompt_tile(1200, 4608, 3584, 1) == (192, 128)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [33, 100, 129, 200, 300])
def test_a_padded_prompt_has_the_same_bits(M):
    """A prompt's products on its own tiles and, padded to its graph's 512 rows, on those of that size."""
    torch.manual_seed(M)
    x = _rand(512, 2048)
    x[M:] = 0
    w, gu = _rand(3072, 2048, scale=0.05), _rand(4096, 2048, scale=0.05)
    ys = [ops.linear_tile(t, w, defer_reduce=True, prompt=True) for t in (x[:M].contiguous(), x)]
    a, b = (y.p.view(y.S, *y.shape) if isinstance(y, ops.SplitK) else y[None] for y in ys)
    assert torch.equal(a, b[:, :M])
    assert torch.equal(ops.linear_tile(x[:M].contiguous(), gu, glu=ops.SILU, prompt=True), ops.linear_tile(x, gu, glu=ops.SILU, prompt=True)[:M])
