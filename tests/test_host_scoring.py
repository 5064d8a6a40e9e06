"""Scoring and context windows on the host (batches of few hits) against the oracle and the GPU forms."""
import random

import numpy as np
import pytest

from operator_amd.engine.match import MatchEngine
from operator_amd.patterns import oracle
from operator_amd.patterns.compiler import compile_patterns
from operator_amd.patterns.synth import LogFactory, synthetic_library


def _hits(eng, rng, docs, n):
    rows = {(rng.randrange(docs), rng.randrange(eng.cp.num_matchers), rng.randrange(60)) for _ in range(n)}
    return np.asarray(sorted(rows), dtype=np.int64).reshape(-1, 3)


@pytest.mark.parametrize("docs,n", [(1, 0), (1, 1), (3, 40), (5, 2000)])
def test_kept_scorer_matches_oracle(docs, n):
    eng = MatchEngine(compile_patterns(synthetic_library(60, seed=2)), device="cpu")
    hits = _hits(eng, random.Random(n), docs, n)
    for _ in range(2):   # the tables are kept, the batch is not
        evs = eng._events_from_hits([b""] * docs, hits)
        for d in range(docs):
            want = oracle.score_doc(eng.cp, {(int(m), int(l)) for i, m, l in hits if i == d})
            assert [(e.pattern, e.line) for e in evs[d]] == [(e.pattern, e.line) for e in want]
            assert [e.score for e in evs[d]] == pytest.approx([e.score for e in want], abs=1e-12)


@pytest.mark.gpu
@pytest.mark.parametrize("docs", [1, 7])
def test_host_and_gpu_forms_agree(docs):
    cp = compile_patterns(synthetic_library(100, seed=0))
    logs = LogFactory(100, seed=4, pool_lines=256).batch(docs, 9000)[0]
    host, gpu = MatchEngine(cp, device="cuda"), MatchEngine(cp, device="cuda", gpu_scorer=True)
    gpu.HOST_CONTEXT_DOCS = 0
    for a, b in zip(host.analyze(logs), gpu.analyze(logs)):
        assert a.summary == b.summary and a.events == b.events
