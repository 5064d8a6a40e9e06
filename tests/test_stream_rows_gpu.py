"""Hyper-connection steps over streams of 128 MiB and more request their rows in groups: the bits of the same rows some hundred at a time, over widths at the
edges of a thread's vectors, stream counts, experts, gates, post norms and chosen rows."""
import pytest
import torch

from operator_amd.ops import decoder as dec

DEV = "cuda"


@pytest.mark.gpu
@pytest.mark.parametrize("S,ld,top,y,gate,post,rows,write", [
    (4, 1032, 2, False, False, False, False, False), (4, 4096, 4, True, True, False, False, True), (3, 2056, 1, False, False, False, False, True),
    (2, 4088, 3, True, False, False, False, True), (8, 1536, 0, True, True, False, False, True), (5, 4096, 2, False, False, False, False, True),
    (1, 4096, 0, True, False, True, False, True), (1, 8192, 2, True, False, True, False, True), (1, 4104, 0, True, False, False, False, True),
    (4, 4096, 2, True, False, False, True, False)])
def test_groups_give_the_same_bits(S, ld, top, y, gate, post, rows, write):
    torch.manual_seed(S + ld)
    T, width = -(-(128 << 20) // (S * ld * 4)) + 3, ld - 8
    rnd = lambda *s: torch.randn(*s, device=DEV)  # noqa: E731
    x, hc, w = rnd(T, S, ld), dec.Stream(rnd(S), rnd(S, S), rnd(S)), rnd(ld)
    yr, g = rnd(T, ld).bfloat16() if y else None, rnd(T) if gate else None
    e, pos = (rnd(T * top + 5, ld).bfloat16(), torch.randperm(T * top, device=DEV).int().view(T, top)) if top else (None, None)
    pw = rnd(ld) if post else None
    pick = torch.randperm(T, device=DEV) if rows else None

    def step(xs, a, b):
        cut = lambda t: None if t is None else t[a:b].contiguous()  # noqa: E731
        o = dec.SublayerOut(y=cut(yr), gate=cut(g), e=e, epos=cut(pos), top=top)
        r = None if pick is None else pick if (a, b) == (0, T) else torch.arange(b - a, device=DEV)
        return dec.stream_step(xs, o, hc, None if rows else hc.inp, w, width, 1e-6, torch.bfloat16, rows=r, write_x=write, post_w=pw)

    whole = x.clone()
    h = step(whole, 0, T)
    if not write:
        assert torch.equal(whole, x)
    for a, b in ((0, 513), (T - 600, T)):   # past 512 rows, whose sums of squares are taken by more threads
        part = x[a:b].clone()
        hp = step(part, a, b)
        assert torch.equal(h[(pick[None] == torch.arange(a, b, device=DEV)[:, None]).int().argmax(1)] if rows else h[a:b], hp)
        assert torch.equal(whole[a:b], part)
