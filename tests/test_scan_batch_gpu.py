"""One-call scan: the report in front of the records, at the edges of the read-back and of the match buffer."""
import numpy as np
import pytest
import torch

from operator_amd import ops
from operator_amd.engine.match import MatchEngine
from operator_amd.patterns.schema import PatternSet

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap", [1, 63, 64, 65, 300])
@pytest.mark.parametrize("nd", [1, 2, 3, 700])
def test_scan_report_edges(nd, cap, monkeypatch):
    monkeypatch.setattr(MatchEngine, "HEAD_MATCHES", 64)
    eng = MatchEngine(PatternSet.from_dicts([{"id": "a", "primary_pattern": {"literal": "refused"}}]), device="cuda", seg_bytes=256)
    for n in (64, 0, 65, 63):                      # records; the buffers of a larger scan are used again
        eng.match_cap = cap
        docs = [(b"\n" * (d % 4) + b"refused" * (n // nd + (d < n % nd)) + b"\nx") for d in range(nd)]
        hits = eng.scan_gpu(docs)
        want = eng.scan_cpu(docs)
        assert len(hits) == n and sorted(map(tuple, hits.tolist())) == sorted(map(tuple, want.tolist()))
        assert eng._doc_newlines[1] == [d.count(b"\n") for d in docs]
        assert hits.dtype == np.int64


def test_nothing_reads_the_buffer_after_an_error(monkeypatch):
    """An error behind the uploads: none of them still reads the pinned buffer when it reaches the caller, and the next scan is right."""
    eng = MatchEngine(PatternSet.from_dicts([{"id": "a", "primary_pattern": {"literal": "refused"}}]), device="cuda", seg_bytes=256)
    docs = [b"refused\n" + b"x" * (1 << 20)] * 256   # 5 ms of upload
    want = eng.scan_gpu(docs)                          # buffers of the size are there
    idle = []

    def fail(*a):
        idle.append(torch.cuda.current_stream().query())   # the uploads are under way
        raise RuntimeError("no memory")

    with monkeypatch.context() as m:
        m.setattr(ops.kernels(), "scan_batch", fail)
        with pytest.raises(RuntimeError, match="no memory"):
            eng._scan_gpu(docs)
        idle.append(torch.cuda.current_stream().query())
    assert idle == [False, True]
    assert np.array_equal(np.sort(eng.scan_gpu(docs), axis=0), np.sort(want, axis=0)) and len(want) == 256
