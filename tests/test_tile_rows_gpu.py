"""Tiles of 96, 128, 160 (gemm_mid), 192, 224 and 256 rows (gemm_tile) sum in the same order, so a plan may take whichever is fastest: the same
bits for every epilogue, at edges of tiles and remainders; and the rule that chooses the rows."""
import pytest
import torch

from operator_amd import ops

DEV = "cuda"


def _rand(*shape, scale=1.0):
    return (torch.randn(*shape, device=DEV) * scale).to(torch.bfloat16)


# one row; a row less and more than a tile of each kind; several rounds of workgroups with a nearly empty last one; the
# shortest K the 256-row tiles take on their persistent schedule, odd numbers of steps
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 128, 128), (95, 272, 192), (97, 256, 320), (161, 1024, 128), (193, 528, 192), (225, 384, 320), (300, 384, 1024), (321, 4224, 192),
                                   (885, 6144, 256), (2600, 16384, 128)])
def test_every_tile_gives_the_same_bits(M, N, K):
    torch.manual_seed(M + N + K)
    C, x, w, b = ops.kernels(), _rand(M, K), _rand(N, K, scale=0.05), _rand(N)
    new = lambda n=N: torch.full((M, n), float("nan"), dtype=torch.bfloat16, device=DEV)  # noqa: E731
    for bias in (None, b):
        C.gemm_tile(x, w, want := new(), bias, 0, 5)
        for rows in (96, 128, 160):
            C.gemm_mid(x, w, y := new(), bias, rows=rows)
            assert torch.equal(y, want), (rows, bias is not None)
    if N % 128 == 0:
        for act in (ops.SILU, ops.GELU_TANH):
            C.gemm_tile(x, w, want := new(N // 2), None, act, 5)
            for rows in (96, 128, 160):
                C.gemm_mid(x, w, y := new(N // 2), None, None, 1, act, rows=rows)
                assert torch.equal(y, want), (rows, act)
    for rows in (192, 224):
        C.gemm_tile(x, w, want := new(), b, 0, 5)
        C.gemm_tile(x, w, y := new(), b, rows=rows)
        assert torch.equal(y, want), rows
        if N % 128 == 0:
            C.gemm_tile(x, w, want := new(N // 2), None, ops.SILU, 5)
            C.gemm_tile(x, w, y := new(N // 2), None, ops.SILU, rows=rows)
            assert torch.equal(y, want), rows
    S = min(3, K // 64)
    slabs = [torch.full((S, M, N), float("nan"), device=DEV) for _ in range(3)]
    for p, rows in zip(slabs, (96, 128, 160)):
        C.gemm_mid(x, w, None, b, p, S, rows=rows)
        assert torch.equal(p, slabs[0])
    r = x.double() @ w.double().t() + b.double()
    mag = x.double().abs() @ w.double().abs().t() + b.double().abs()
    assert ((slabs[0].double().sum(0) - r).abs() <= K * 2.0 ** -24 * mag).all()   # fp32 sums of K terms


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 200, 256, 257])
def test_operands_off_their_alignment(M):
    """Biases off 16 bytes come as a copy, outputs run on the kernels with narrower stores: the same bits."""
    torch.manual_seed(M)
    x, w, b = _rand(M, 256), _rand(512, 256, scale=0.05), _rand(512)
    want = ops.linear_tile(x, w, bias=b)
    off = torch.cat([b[:1], b])[1:]
    wide = torch.zeros(M, 524, dtype=torch.bfloat16, device=DEV)
    assert off.data_ptr() % 16 and torch.equal(ops.linear_tile(x, w, bias=off), want)
    assert torch.equal(ops.linear_tile(x, w, wide[:, 4:516], bias=b), want) and not wide[:, :4].any() and not wide[:, 516:].any()


@pytest.mark.gpu
@pytest.mark.parametrize("M,rows", [(1, 256), (256, 256), (257, 256), (200, 192), (300, 224)])
def test_bias_off_its_alignment_is_copied(M, rows):
    """The epilogues load a bias 16 (8) bytes at a time: one off that alignment is read from an aligned copy, whatever the tile."""
    torch.manual_seed(M)
    C, x, w, b = ops.kernels(), _rand(M, 256), _rand(512, 256, scale=0.05), _rand(512)
    y, want = (torch.empty(M, 512, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    made = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]  # noqa: E731
    n = made()
    C.gemm_tile(x, w, want, b, rows=rows)
    assert made() == n
    for shift in (1, 4):   # 2 and 8 bytes
        off = torch.cat([b[:shift], b])[shift:]
        n = made()
        C.gemm_tile(x, w, y.zero_(), off, rows=rows)
        assert made() == n + 1 and torch.equal(y, want)


def test_rows_that_the_kernels_have():
    for N, K in ((16, 128), (272, 192), (4096, 4096), (28672, 4096), (3584, 18944)):
        for M in (1, 128, 129, 300, 885, 4096, 30000):
            assert ops.tile_rows(M, N, K, 2) in (96, 128, 160)
            assert ops.tile_rows(M, N, K) in (96, 128, 160, 192, 224, 256)
    assert ops.tile_rows(100, 6144, 4096) == 128
    assert [ops.tile_rows(885, 6144, 4096), ops.tile_rows(300, 28672, 4096), ops.tile_rows(28000, 4096, 14336)] == [96, 160, 256]


def test_one_round_has_no_stores_between_rounds():
    """Tiles that come in one round of workgroups cost their steps alone: the smaller ones win (257 rows of 3072 x 2048 in 3 slices:
    13.7 us on 96 rows, 18.4 on 160; 385 rows of 768 x 4096 in 8 12.1 and 15.8)."""
    assert all(ops.tile_rows(*a) == 96 for a in ((257, 3072, 2048, 3), (300, 2048, 2048, 4), (385, 768, 4096, 8), (160, 3584, 4096, 4), (129, 3584, 4096, 4)))


# the smallest vocabulary of more than a round of 256-column tiles; rows at the edges of the rule
@pytest.mark.gpu
@pytest.mark.parametrize("K,Ms", [(4096, (129, 256)), (8192, (208, 209))])
def test_wide_vocabularies_give_the_same_bits_on_either_schedule(K, Ms):
    torch.manual_seed(K)
    w, x = _rand(65552, K, scale=0.05), _rand(256, K)
    for M in Ms:
        ops.kernels().gemm_tile(x[:M], w, want := torch.full((M, 65552), float("nan"), dtype=torch.bfloat16, device=DEV), None, 0, 5)
        assert torch.equal(ops.linear_tile(x[:M], w), want)


def test_schedule_of_wide_vocabularies():
    assert all(ops.loose_tiles(M, 128256, 4096) for M in (129, 192, 256)) and ops.loose_tiles(256, 128256, 8192)
    assert not any(ops.loose_tiles(*a) for a in ((128, 128256, 4096), (257, 128256, 4096), (192, 128256, 8192), (256, 152064, 3584),
                                                 (256, 32768, 4096), (256, 151936, 2048)))


@pytest.mark.gpu
def test_rows_longer_than_a_buffer_bound():
    """256 weight rows of 2^23 columns are 4 GiB, past the 32 bits of the persistent schedule's buffer bounds: such products run on the
    kernel with 64-bit addresses. Small whole numbers: every sum is exact in fp32, whatever its order."""
    if torch.cuda.get_device_properties(0).total_memory < 32 << 30:
        pytest.skip("needs 20 GB")
    K, M, N, step = 1 << 23, 3, 256, 1 << 19
    torch.manual_seed(0)
    w, x = torch.empty(N, K, dtype=torch.bfloat16, device=DEV), torch.empty(M, K, dtype=torch.bfloat16, device=DEV)
    want = torch.zeros(M, N, device=DEV)
    for k in range(0, K, step):
        w[:, k:k + step] = torch.randint(-1, 2, (N, step), device=DEV, dtype=torch.int8)
        x[:, k:k + step] = torch.randint(-1, 2, (M, step), device=DEV, dtype=torch.int8)
        want += x[:, k:k + step].float() @ w[:, k:k + step].float().t()
    assert want.abs().max() < 1 << 24
    y = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    ops.kernels().gemm_tile(x, w, y)
    assert torch.equal(y, want.bfloat16())
    assert torch.equal(ops.linear_tile(x, w), y)
    with pytest.raises(RuntimeError):
        ops.kernels().gemm_tile(x, w, y, rows=192)
