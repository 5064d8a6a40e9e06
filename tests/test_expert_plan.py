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
