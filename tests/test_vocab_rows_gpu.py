"""Vocabularies of 9 to 127 rows on a part of a decode bucket's row tile: the bits of the whole tile, nothing written behind the last row, what a part is refused
with, and the rule that takes it."""
import pytest
import torch

from operator_amd import ops

DEV = "cuda"


def _rand(*shape):
    return torch.randn(*shape, device=DEV).to(torch.bfloat16)


# K of one step, fewer than the ring's, of steps that start apart (2048, 4096)
@pytest.mark.gpu
@pytest.mark.parametrize("N,K", [(29568, 64), (32000, 192), (33024, 2048), (32768, 4096)])
def test_parts_of_a_tile(N, K):
    torch.manual_seed(K)
    x, w = _rand(128, K), _rand(N, K) * 0.05
    for bm in (64, 128):
        _, bn, _, ns = ops.gemm_plan(bm, N, K, False)[:4]
        whole = torch.empty(bm, N, dtype=torch.bfloat16, device=DEV)
        ops.kernels().gemm_decode(x[:bm], w, whole, None, 1, bn, bm, False, False, ns)
        for M in (9, 16, 33, 63) if bm == 64 else (65, 127):
            guard = torch.full((M + 1, N), float("nan"), dtype=torch.bfloat16, device=DEV)
            ops.kernels().gemm_decode(x[:M], w, guard[:M], None, 1, bn, bm, False, False, ns)
            assert torch.equal(guard[:M], whole[:M]) and guard[M].isnan().all(), M
            assert torch.equal(ops.linear(x[:M], w), whole[:M]), M
    # one rounding to bf16 of an fp32 sum
    r, bound = (f(x[:100].double()) @ f(w.double()).t() for f in (lambda t: t, torch.abs))
    assert ((ops.linear(x[:100], w).double() - r).abs() <= 2.0 ** -8 * r.abs() + K * 2.0 ** -24 * bound).all()


@pytest.mark.gpu
def test_other_parts_are_refused():
    x, w, y = _rand(70, 128), _rand(512, 128), torch.empty(70, 512, dtype=torch.bfloat16, device=DEV)
    p = torch.empty(2 * 70 * 512, device=DEV)
    for bm, S, glu in ((64, 1, 0), (128, 2, 0), (128, 1, 1)):
        with pytest.raises(RuntimeError):
            ops.kernels().gemm_decode(x, w, y[:, :256].contiguous() if glu else y, p, S, 128, bm, glu, False, 3)


def test_the_rule():
    assert [ops.vocab_rows_plan(M, 128256, 4096) for M in (8, 9, 63, 64, 65, 127)] == [None, (64, 128, 1, 3), (64, 128, 1, 3), None, None, None]
    assert ops.vocab_rows_plan(100, 32000, 2048)[:3] == (128, 128, 1) and ops.vocab_rows_plan(20, 32000, 2048)[:3] == (64, 128, 1)
    # fewer tiles than CUs, columns that are no whole tiles, K of a part of a step
    assert not any(ops.vocab_rows_plan(20, N, K) for N, K in ((16128, 4096), (32064, 2048), (32000, 2080)))
