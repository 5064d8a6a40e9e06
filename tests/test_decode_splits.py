"""Splits of decode attention: buckets that are full or nearly so have what their size gives, a bucket of few sequences is cut further, and an engine captures
every count that its buckets can ask for."""
import pytest

from operator_amd import ops
from operator_amd.engine.llm import LLMEngine, _buckets


@pytest.mark.parametrize("hkv", [1, 2, 4, 8])
@pytest.mark.parametrize("least", [None, 128])
def test_rows_of_a_bucket(hkv, least):
    b = _buckets(256)
    for lo, bp in zip([0] + b, b):
        for n in range(lo + 1, bp + 1):
            for ctx in (100, 300, 1000, 4000):
                whole, s = (ops.decode_splits(ctx, bp, hkv, least, r) for r in (None, n))
                assert s >= whole and s & (s - 1) == 0 and (s == whole or (s * n * hkv <= ops.DECODE_TARGET_BLOCKS and s <= -(-ctx // (least or ops.DECODE_MIN_SPLIT_TOKENS))))
                if bp <= 8 or n > bp // 2:
                    assert s == whole, (bp, n)
    assert [ops.decode_splits(4000, 64, 4, None, n) for n in (9, 16, 17, 32, 33, 64)] == [4, 4, 2, 2, 1, 1]


@pytest.mark.parametrize("most", [1, 8, 16, 48, 64, 256])
@pytest.mark.parametrize("hkv", [1, 4, 8])
def test_every_count_is_captured(most, hkv):
    class Model:
        split_tokens = 128 if hkv == 1 else None

    eng = LLMEngine.__new__(LLMEngine)
    eng.buckets, eng.hkv, eng.model, eng.max_context = _buckets(most), hkv, Model(), 8192
    for n in range(1, most + 1):
        bp = eng._bucket(n)
        assert {eng._splits(ctx, bp, n) for ctx in range(1, 8193, 61)} <= set(eng.split_options(bp)), n
