"""gemm_mid (128 x 256 tiles, K slices): tails, every epilogue, slices by the reduce pass and by the consumer, several
rounds of tiles per workgroup, against fp64; and the plan that chooses it."""
import pytest
import torch

from operator_amd import ops
from operator_amd.ops import reference as ref

DEV = "cuda"


def _rand(*shape, scale=1.0):
    return (torch.randn(*shape, device=DEV) * scale).to(torch.bfloat16)


def _check(y, r, mag, K, extra=0.0):
    """bf16 rounding of the result (2^-8 of it) plus fp32 accumulation (K 2^-24 of the sum of magnitudes)."""
    assert ((y.double() - r).abs() <= (2.0 ** -8 + extra) * r.abs() + K * 2.0 ** -24 * mag + 1e-30).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,S", [
    (1, 16, 64, 1), (127, 272, 128, 2), (128, 256, 192, 3), (129, 528, 1024, 5), (300, 4096, 2048, 16), (885, 4096, 1088, 2),
    (700, 16384, 128, 1), (700, 16400, 192, 1), (2300, 8192, 64, 1), (130, 48000, 128, 2)])
def test_gemm_mid(M, N, K, S):
    torch.manual_seed(M + N + K)
    x, w, b = _rand(M, K), _rand(N, K, scale=0.05), _rand(N, scale=0.5)
    r, mag = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    nan = lambda *s, dt=torch.float32: torch.full(s, float("nan"), dtype=dt, device=DEV)  # noqa: E731
    y = nan(M, N, dt=torch.bfloat16)
    ops.kernels().gemm_mid(x, w, y, None, nan(S, M, N), S)
    _check(y, r, mag, K)
    if S > 1:
        slabs = nan(S, M, N)
        ops.kernels().gemm_mid(x, w, None, None, slabs, S)
        assert ((slabs.double().sum(0) - r).abs() <= K * 2.0 ** -24 * mag).all()
        return
    ops.kernels().gemm_mid(x, w, y, b)
    _check(y, r + b.double(), mag + b.double().abs(), K)
    wide = nan(M, N + 64, dt=torch.bfloat16)
    ops.kernels().gemm_mid(x, w, wide[:, 32:32 + N])
    _check(wide[:, 32:32 + N], r, mag, K)
    assert wide[:, :32].isnan().all() and wide[:, 32 + N:].isnan().all()


@pytest.mark.gpu
@pytest.mark.parametrize("act", [ops.SILU, ops.GELU_TANH])
@pytest.mark.parametrize("M,inter,K,S", [(33, 128, 128, 2), (200, 8192, 192, 1), (520, 8256, 256, 1)])
def test_gemm_mid_gated(M, inter, K, S, act):
    torch.manual_seed(M + K)
    x, g, u = _rand(M, K), _rand(inter, K, scale=0.05), _rand(inter, K, scale=0.05)
    y = torch.full((M, inter), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.kernels().gemm_mid(x, ops.interleave_gate_up(g, u), y, None, torch.empty(S, M, 2 * inter, device=DEV), S, act)
    gate, up = ((x.double() @ w.double().t()).to(torch.bfloat16) for w in (g, u))
    r = ref.silu_mul(torch.cat([gate, up], 1), None, act == ops.GELU_TANH).double()
    # each of gate, act(gate) and up may round the other way (2^-8; the activation's slope is below 1.2),
    # and a gate near 0 carries its absolute error
    assert ((y.double() - r).abs() <= 5 * 2.0 ** -8 * r.abs() + 2.0 ** -8 * 1.2 * up.double().abs() * gate.double().abs() + 1e-6).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,S", [(1, 16, 128, 2), (130, 272, 448, 3), (300, 4608, 3584, 2)])
def test_bias_is_in_the_first_slab(M, N, K, S):
    torch.manual_seed(M + N)
    x, w, b = _rand(M, K), _rand(N, K, scale=0.05), _rand(N, scale=0.5)
    r = x.double() @ w.double().t() + b.double()
    mag = x.double().abs() @ w.double().abs().t() + b.double().abs()
    y, slabs = torch.empty(M, N, dtype=torch.bfloat16, device=DEV), torch.full((S, M, N), float("nan"), device=DEV)
    ops.kernels().gemm_mid(x, w, y, b, slabs, S)
    _check(y, r, mag, K)
    for y in (ops.linear(x, w, bias=b), ops.linear(x, w, bias=b, defer_reduce=True)):
        if isinstance(y, ops.SplitK):
            y = y.p[:y.S * M * N].view(y.S, M, N).sum(0)
        _check(y, r, mag, K)


def test_mid_plan_is_launchable():
    """Every plan is one gemm_mid takes, padded batches keep their plan, large products keep the 256-row tiles."""
    for N, K in ((16, 128), (272, 192), (4096, 4096), (4096, 14336), (28672, 4096), (128256, 4096), (151936, 2048)):
        for defer in (False, True):
            for M in (1, 2, 31, 33, 127, 128, 129, 257, 885, 2047, 4096, 9999, 28000):
                S = ops.mid_plan(M, N, K, defer)
                assert S is None or 1 <= S <= min(16, K // 64)
                assert ops.mid_plan(M, N, K, defer, False) in (None, 1)
            assert ops.mid_plan(322, N, K, defer) == ops.mid_plan(512, N, K, defer)
            for M in (33, 64, 65, 100, 127, 129, 200, 255):   # a prompt, in its graph one of 512 rows
                if N < ops.LM_HEAD_MIN_N:
                    assert ops.mid_plan(M, N, K, defer, prompt=True) == ops.mid_plan(512, N, K, defer)
                else:   # the 512-row plan is the 256-row tiles over the whole K: no slices
                    assert ops.mid_plan(M, N, K, defer, prompt=True) in (None, 1) and ops.mid_plan(512, N, K, defer) is None
    assert ops.mid_plan(28000, 4096, 14336, True) is None
    assert ops.mid_plan(885, 4096, 14336, True) == 2
    # a decode batch of the same rows is not padded: slices that fill the GPU
    assert ops.mid_plan(100, 4096, 14336, True) == 14 > ops.mid_plan(100, 4096, 14336, True, prompt=True) == 4


def test_fp32_prompts_take_their_graphs_slices():
    for M in (33, 100, 255, 256, 500, 512):
        assert ops.f32_plan_rows(M, True) == 512 and ops.f32_plan_rows(M, False) == M
    assert ops.f32_plan_rows(513, True) == 1024 and ops.f32_plan_rows(32, True) == 32


@pytest.mark.parametrize("M,N,K,wide", [(1, 4096, 4096, 8192), (1, 272, 1024, 288), (1, 4096, 4096, 4096), (40, 4096, 4096, 8192)])
def test_rows_of_a_wider_output_are_not_sliced(monkeypatch, M, N, K, wide):
    """The reduce pass of K slices writes its rows back to back: one row out of a wider buffer is contiguous for torch,
    but its row stride is the buffer's, which the kernel takes in one slice only."""
    seen = []

    class Kernels:
        def gemm_mid(self, x, w, y, bias, part, S, glu=0):
            seen.append((S, y.stride(0)))

        def gemm_tile(self, x, w, y, bias, glu):
            seen.append((1, y.stride(0)))

    monkeypatch.setattr(ops, "kernels", Kernels)
    x, w, b = (torch.zeros(s, dtype=torch.bfloat16) for s in ((M, K), (N, K), (N,)))
    out = torch.zeros(M, wide, dtype=torch.bfloat16)[:, :N]
    ops.linear_tile(x, w, out, b)
    assert seen[0][1] == wide and (seen[0][0] == 1 or wide == N)
    assert (seen[0][0] > 1) == (wide == N)


@pytest.mark.gpu
def test_one_row_into_a_wider_output():
    torch.manual_seed(1)
    x, w, b = _rand(1, 4096), _rand(4096, 4096, scale=0.05), _rand(4096)
    buf = torch.full((3, 8192), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.linear(x, w, out=buf[:1, :4096], bias=b)
    _check(buf[:1, :4096], x.double() @ w.double().t() + b.double(), x.double().abs() @ w.double().abs().t() + b.double().abs(), 4096)
    assert buf[0, 4096:].isnan().all() and buf[1:].isnan().all()


def test_a_measured_entry_of_few_rows_wins(monkeypatch):
    assert ops._mid_beats_skinny(32, 4096, 14336, True)
    monkeypatch.setitem(ops._gemm_table_get(), ("skinny", 32, 4096, 14336), 8)
    assert not ops._mid_beats_skinny(32, 4096, 14336, True) and ops.skinny_plan(32, 4096, 14336) == 8


@pytest.mark.gpu
@pytest.mark.parametrize("dx,dw,kernel", [(0, 0, "gemm_mid"), (1, 0, "gemm_skinny"), (0, 4, "gemm_skinny"), (8, 8, "gemm_mid")])
def test_few_rows_off_their_alignment_stay_on_plain_loads(monkeypatch, dx, dw, kernel):
    """gemm_mid stages 16-B pieces by LDS-DMA; gemm_skinny's loads take operands at any address. Nothing is launched."""
    M, N, K = 24, 4096, 14336
    seen = []

    class Kernels:
        def __getattr__(self, name):
            return lambda *a: seen.append(name)

    monkeypatch.setattr(ops, "kernels", Kernels)
    x, w = (torch.empty(n * K + 8, dtype=torch.bfloat16, device=DEV)[d:d + n * K].view(n, K) for n, d in ((M, dx), (N, dw)))
    for defer in (False, True):
        ops.linear(x, w, defer_reduce=defer)
    assert seen == [kernel] * 2


def test_few_rows_leave_gemm_skinny_where_it_was_measured_slower():
    """Both sides were timed at these shapes (rows, N, K, deferred): none of the first is faster in gemm_mid."""
    for M, N, K, defer in ((17, 3072, 3072, True), (24, 2560, 2048, True), (32, 2048, 2048, True), (17, 4096, 4096, True),
                           (17, 2048, 8192, True), (5, 32768, 4096, False), (8, 32768, 4096, False), (6, 151936, 2048, False),
                           (5, 64128, 4096, False), (5, 128256, 2048, False)):
        assert not ops._mid_beats_skinny(M, N, K, defer), (M, N, K, defer)
    for M, N, K, defer in ((17, 4096, 14336, True), (24, 3584, 3584, True), (32, 6144, 4096, False), (5, 128256, 3072, False),
                           (6, 128256, 8192, False), (5, 152064, 3584, False), (8, 128256, 4096, False), (16, 32768, 4096, False)):
        assert ops._mid_beats_skinny(M, N, K, defer), (M, N, K, defer)


def test_gemm_splits_is_still_there():
    from operator_amd.ops import gemm_splits

    assert [gemm_splits(64, n, k) for n, k in ((4096, 14336), (4096, 192), (16384, 4096), (8192, 4096), (64, 8192))] == [4, 1, 1, 2, 8]
