"""decode_advance with sampling candidates and a page table: the tokens of the sampler's own merge, the state of the plain advance, and the
slots and sampler positions that decode_slots has of the state it leaves."""
import pytest
import torch

from operator_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _state(B, MP, P, ms):
    bt = torch.randint(0, 5000, (B, MP), dtype=torch.int32, device=DEV)
    ctx = torch.randint(1, MP * P + 1, (B,), dtype=torch.int32, device=DEV)   # the last one steps past its table
    ctx[::5] = 0
    if B > 1:
        ctx[1] = P   # its next token opens a page
    z = lambda *s: torch.zeros(*s, dtype=torch.long, device=DEV)  # noqa: E731
    return dict(ids=z(B), hist=z(B, ms), pos=(ctx.long() - 1).clamp_min(0), ctx=ctx, step=torch.tensor([11], device=DEV)), bt


# one row, rows in one workgroup each (224 and more, short vocabularies), odd part counts
@pytest.mark.parametrize("B,V", [(1, 128256), (7, 32000), (64, 32000), (130, 28672), (223, 98304), (225, 98304), (3, 1000), (1024, 512)])
def test_candidates_and_slots(B, V):
    torch.manual_seed(B)
    P, MP, ms = 16, 9, 4
    st, bt = _state(B, MP, P, ms)
    x = torch.randn(B, V, device=DEV).bfloat16()
    x[0, V // 2:] = x[0, :V - V // 2]   # equal values: the smaller column
    temp = torch.rand(B, device=DEV)
    temp[::3] = 0.0
    temp.view(torch.int32)[2::7] = ops.NO_SAMPLE_BITS
    seeds, spos = torch.arange(B, device=DEV) + 3, torch.randint(0, 4000, (B,), device=DEV)
    if B > 3:
        x[3] = float("-inf")   # nothing to choose from
        temp[3] = 0.5
    want = {k: t.clone() for k, t in st.items()}
    ops.kernels().decode_advance(ops.sample(x, temp, seeds, spos), **want)
    ws, wp = torch.empty_like(spos), torch.empty_like(spos)
    ops.kernels().decode_slots(bt, want["pos"], want["ctx"], ws, wp, P)
    cand = ops.sample_candidates(x, temp, seeds, spos)
    assert (cand["tok"] is None) == (ops.kernels().sample_parts(B, V) > 1)
    slots, nxt = torch.full_like(spos, -7), torch.full_like(spos, -7)
    ops.kernels().decode_advance(**st, bt=bt, slots=slots, spos=nxt, page_size=P, **cand)
    assert all(torch.equal(st[k], want[k]) for k in st)
    assert torch.equal(slots, ws) and torch.equal(nxt, wp)


def test_refusals():
    st, bt = _state(4, 3, 16, 2)
    tok, t = torch.zeros(4, dtype=torch.long, device=DEV), torch.zeros(4, device=DEV)
    part, s = torch.zeros(4, 2, 2, device=DEV), torch.zeros(4, dtype=torch.long, device=DEV)
    for bad in (dict(tok=None), dict(tok=tok, part=part, temperature=t), dict(tok=None, part=part), dict(tok=None, part=part[:3], temperature=t),
                dict(tok=tok[:3]), dict(tok=tok, bt=bt), dict(tok=tok, bt=bt, slots=s, spos=s, page_size=0), dict(tok=tok, bt=bt[:2], slots=s, spos=s, page_size=16)):
        with pytest.raises(RuntimeError):
            ops.kernels().decode_advance(**st, **bad)


# several workgroups a row and one; rows off 16 bytes, vocabularies that are no multiple of 4 or 8; given rows beside sampled ones
@pytest.mark.parametrize("B,V,ld", [(1, 128256, 128256), (6, 32000, 32008), (5, 32004, 32004), (3, 16387, 16400), (230, 1001, 1001), (9, 4096, 4100), (256, 20001, 20008)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_given_rows_leave_through_the_sampler(B, V, ld, dtype):
    torch.manual_seed(B + V)
    x = torch.randn(B, ld, device=DEV).to(dtype)[:, :V]
    temp = torch.full((B,), 0.7, device=DEV)
    temp.view(torch.int32)[:] = torch.where(torch.arange(B, device=DEV) % 4 == 3, temp.view(torch.int32), ops.NO_SAMPLE_BITS)
    seeds, spos = torch.arange(B, device=DEV), torch.arange(B, device=DEV) + 9
    n = B + 2
    dst = torch.randperm(n, device=DEV, dtype=torch.int32)[:B]
    dst[B // 2] = -1 if B % 2 else n   # to no row
    for off in (0, 1):   # the output's address off 16 bytes
        flat = torch.full((n * V + 8,), float("nan"), device=DEV)
        out = flat[off:off + n * V].view(n, V)
        given = torch.tensor([out.data_ptr(), n], device=DEV)
        st, _ = _state(B, 2, 16, 4)
        cand = ops.sample_candidates(x, temp, seeds, spos, given, dst)
        ops.kernels().decode_advance(**st, given=given, **cand)
        want = torch.full((n, V), float("nan"), device=DEV)
        for r in range(B):
            if r % 4 != 3 and 0 <= dst[r] < n:
                want[dst[r]] = x[r].float()
        assert torch.equal(out.nan_to_num(7.5), want.nan_to_num(7.5)) and flat[off + n * V:].isnan().all() and flat[:off].isnan().all()
        assert torch.equal(st["ids"], ops.sample(x, temp, seeds, spos))
        assert given.tolist() == [0, n]   # and no later step writes there
        flat.fill_(1.0)
        ops.sample_candidates(x, temp, seeds, spos, given, dst)
        assert (flat == 1.0).all()
