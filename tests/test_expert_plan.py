"""The lines between the forms of the experts' products."""
from operator_amd.ops import decoder as dec


def test_plan():
    for weights in (1 << 21, 1 << 24, 1 << 26):
        for tiles in (True, False):
            forms = [dec.expert_plan(s, 8, weights, tiles) for s in range(1, 4000)]
            assert forms == sorted(forms, key=lambda p: p)          # more rows, larger tiles
            assert forms[0] == 0 and forms[-1] == 256
            assert tiles or set(forms) == {0, 256}
    assert dec.expert_plan(2 * dec.MOE_LIST_MAX_SLOTS, 8192) == 64   # more slots than a workgroup lists
    assert dec.expert_plan(20, 8, 1 << 22, False) == 0 and dec.expert_plan(24, 8, 1 << 22) == 64


def test_small_experts_and_few_tiles_keep_their_lists():
    plan = lambda rows, E, ld, ff: dec.expert_plan(rows * E, E, ld * ff, True, min(ld, 2 * ff))  # noqa: E731
    for E, ld, ff in ((8, 2048, 2048), (4, 2176, 320), (16, 2304, 512), (8, 1280, 1408), (4, 4096, 4096), (2, 8192, 4096), (64, 512, 704)):
        assert [plan(r, E, ld, ff) for r in (1, 3, 5, 7, 8)] == [0, 0, 0, 0, 64]
    for E, ld, ff in ((8, 4096, 4096), (32, 2048, 1024), (64, 2048, 1024), (16, 4096, 1024), (8, 4096, 14336), (4, 8192, 4096)):
        assert [plan(r, E, ld, ff) for r in (2, 3, 7)] == [0, 64, 64]
