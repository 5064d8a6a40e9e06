"""Scoring and context windows on the host (batches of few hits) against the oracle and the GPU forms."""
import random

import numpy as np
import pytest
import torch

from operator_amd.engine.match import MatchEngine
from operator_amd.ops import patterns
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


def test_score_events_takes_longer_tables():
    """The tables' extra entries are not read; missing ones are refused, not read past the end."""
    P = patterns()
    hits, m = ([0, 0, 0], [0, 1, 1], [4, 6, 9]), 2
    exact = ([0], [0.5], [3], [[1]], [[2.0]], [[10]])
    longer = ([0], [0.5, 9.0], [3, 1], [[1], [0]], [[2.0, 7.0], []], [[10, 1], [5]])
    want = P.score_events(*hits, 1, *exact, m)
    assert len(want[0]) == 1 and P.score_events(*hits, 1, *longer, m) == want
    for i in range(1, 6):
        short = list(exact)
        short[i] = [] if i < 4 else [[]]
        with pytest.raises(ValueError):
            P.score_events(*hits, 1, *short, m)


@pytest.mark.parametrize("native,gpu_scorer,n,on_gpu", [
    (True, None, 0, False), (True, None, MatchEngine.HOST_SCORE_HITS, False), (True, None, MatchEngine.HOST_SCORE_HITS + 1, True),
    (False, None, 1, True), (True, True, 1, True), (False, True, 1, True), (True, False, 9999, False), (False, False, 9, False)])
def test_where_a_gpu_engine_scores(monkeypatch, native, gpu_scorer, n, on_gpu):
    """Few hits go to the native scorer; without it, or where the GPU scorer is asked for, they are the GPU's."""
    eng = MatchEngine(compile_patterns(synthetic_library(20, seed=2)), device="cpu", use_native_scorer=native, gpu_scorer=gpu_scorer)
    if gpu_scorer is None:
        eng.gpu_scorer = True   # what an engine on the GPU sets
    monkeypatch.setattr(eng, "device", torch.device("cuda"))
    monkeypatch.setattr(eng, "_events_gpu", lambda hits, docs: "gpu")
    hits = np.stack([np.zeros(n, np.int64), np.zeros(n, np.int64), np.arange(n)], 1)
    assert (eng._events_from_hits([b""], hits) == "gpu") == on_gpu


@pytest.mark.gpu
@pytest.mark.parametrize("docs", [1, 7])
def test_host_and_gpu_forms_agree(docs):
    cp = compile_patterns(synthetic_library(100, seed=0))
    logs = LogFactory(100, seed=4, pool_lines=256).batch(docs, 9000)[0]
    host, gpu = MatchEngine(cp, device="cuda"), MatchEngine(cp, device="cuda", gpu_scorer=True)
    gpu.HOST_CONTEXT_DOCS = 0
    for a, b in zip(host.analyze(logs), gpu.analyze(logs)):
        assert a.summary == b.summary and a.events == b.events


@pytest.mark.gpu
def test_gpu_scorer_alone():
    """Without the native scorer the GPU scores every batch, one without hits among them."""
    cp = compile_patterns(synthetic_library(100, seed=0))
    logs = LogFactory(100, seed=4, pool_lines=256).batch(3, 9000)[0]
    alone, host = MatchEngine(cp, device="cuda", use_native_scorer=False), MatchEngine(cp, device="cpu")
    for docs in ([b"zzz\n", b""], logs):
        for a, b in zip(alone.analyze(docs), host.analyze(docs)):
            assert a.summary == b.summary and a.events == b.events


@pytest.mark.gpu
def test_default_engine_on_both_sides_of_the_host_threshold(monkeypatch):
    """The same logs' events with as many hits as the host takes, and with one more."""
    cp = compile_patterns(synthetic_library(100, seed=0))
    eng, host = MatchEngine(cp, device="cuda"), MatchEngine(cp, device="cpu")
    scored = []
    monkeypatch.setattr(eng, "_events_gpu", lambda hits, docs, f=eng._events_gpu: scored.append(len(hits)) or f(hits, docs))
    rng, n = random.Random(3), MatchEngine.HOST_SCORE_HITS
    for extra in (0, 1):
        rows = set()
        while len(rows) < n + extra:
            rows.add((rng.randrange(7), rng.randrange(cp.num_matchers), rng.randrange(400)))
        hits = np.asarray(sorted(rows), dtype=np.int64)
        got, want = (e._events_from_hits([b""] * 7, hits) for e in (eng, host))
        for a, b in zip(got, want):
            # an fp64 score is a dozen roundings of 2^-53 each, fused on the GPU; scores that differ so little may swap places
            assert sorted((e.pattern, e.line) for e in a) == sorted((e.pattern, e.line) for e in b)
            assert [e.score for e in a] == pytest.approx([e.score for e in b], rel=1e-14)
    assert scored == [n + 1]
