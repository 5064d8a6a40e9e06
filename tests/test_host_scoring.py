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


def _plain(results):
    """Everything a result holds but its id, its processing time and the object identities."""
    out = []
    for r in results:
        for m in (r, r.summary, *r.events):
            assert m.__pydantic_fields_set__ == set(type(m).model_fields) and m.__pydantic_extra__ == {} and m.__pydantic_private__ is None
            assert list(m.__dict__) == list(type(m).model_fields)
        o = r.model_dump()
        assert len(o.pop("analysis_id")) == 36 and o["metadata"].pop("processingTimeMs") >= 0
        out.append(o)
    return out


@pytest.mark.parametrize("max_events", [0, 2, 50])
@pytest.mark.parametrize("lazy", [False, True])
def test_native_results_equal_those_built_in_python(lazy, max_events):
    cp = compile_patterns(synthetic_library(60, seed=2))
    docs = LogFactory(60, seed=3, pool_lines=256).batch(6, 9000)[0]
    docs += [b"", b"\n", docs[0].rstrip(b"\n"), docs[1].replace(b"\n", b"\r\n"), docs[2][:2000] + b"\xff\xfe\n" + docs[2][2000:], docs[3] + docs[3]]
    native, plain = (MatchEngine(cp, device="cpu", use_native_scorer=n, max_events=max_events) for n in (True, False))
    for pods in (None, [(f"pod-{i}", "ns") for i in range(len(docs))]):
        a, b = (e.analyze(docs, pods, lazy=lazy) for e in (native, plain))
        assert _plain(a) == _plain(b)
    assert any(r.events for r in a) == (max_events > 0) and len({r.analysis_id for r in a}) == len(docs)
    assert _plain(native.analyze(tuple(docs))) == _plain(plain.analyze(docs))
    assert native.analyze([]) == [] == plain.analyze([])


def test_result_batch_refuses_what_does_not_fit():
    P, eng = patterns(), MatchEngine(compile_patterns(synthetic_library(20, seed=2)), device="cpu")
    eng.analyze([b"x\n"])
    hits = np.asarray([[0, int(eng.cp.pattern_primary[0]), 0, 3]], dtype=np.int64)
    ok = ([b"abc def\n"], hits, 50, 0.5, bytes(16))
    for i, bad in ((0, ["text"]), (1, hits[:, :3]), (1, hits + [[1, 0, 0, 0]]), (4, bytes(15))):
        with pytest.raises((TypeError, ValueError, IndexError)):
            P.ResultBatch(eng._tables, *ok[:i], bad, *ok[i + 1:])
    b = P.ResultBatch(eng._tables, *ok)
    assert b.queries().tolist() == [[0, 3, 3]]
    with pytest.raises(RuntimeError):
        b.build(0, None, None, 0, 1.0)
    for bad in (np.zeros((0, 4), np.int64), np.asarray([[0, 9, 0, 7]]), np.asarray([[3, 7, 0, 7]])):
        with pytest.raises((ValueError, IndexError)):
            b.windows(bad)
    b.windows(np.asarray([[0, 7, 0, 7]]))
    r = b.build(0, "p", "n", 1, 2.0)
    assert r.events[0].context == ["abc def"] and r.events[0].matched_line == "abc def" and r.metadata["totalLines"] == 2
    with pytest.raises(IndexError):
        b.build(1, None, None, 0, 1.0)


@pytest.mark.parametrize("rx,line", [(rb"^ab", b"xab"), (rb"^ab", b"ab"), (rb"a*$", b"bb"), (rb"abc\b", b"zabc abcd"), (rb"aab", b"aaab"), (rb"\Bb", b"ab"),
                                     (rb"abab(c|$)", b"abaabab"), (rb"a.c", b"aac"), (rb"(^|x)y", b"ay xy"), (rb"abcd", b"abc"), (rb"b", b"")])
def test_search_passes_over_bytes_no_match_starts_at(rx, line):
    import re

    from operator_amd.patterns.nfa import compile_nfa

    prog = compile_nfa(rx, 0)
    assert prog is not None
    assert patterns().RegexSet([prog]).search(0, line) == (re.search(rx, line) is not None)


def test_large_results_leave_the_lock_to_other_threads():
    """Scoring, context lines and result objects of a large batch take a tenth of a second and more: another thread runs in between, not behind."""
    import gc
    import threading
    import time

    eng = MatchEngine(compile_patterns(synthetic_library(200, seed=2)), device="cpu", max_events=1000)
    eng.analyze([b"x\n"])
    rng = np.random.default_rng(0)
    lines, per, n = 5000, 1000, 64
    doc = b"".join(b"line %05d " % i + b"x" * 50 + b"\n" for i in range(lines))
    rows = np.concatenate([np.stack([np.full(per, d), rng.choice(eng.cp.pattern_primary, per), rng.choice(lines, per, replace=False), np.zeros(per)], 1)
                           for d in range(n)]).astype(np.int64)
    rows[:, 3] = rows[:, 2] * (len(doc) // lines)
    stop, ticks = threading.Event(), []

    def tick():
        while not stop.is_set():
            ticks.append(time.perf_counter())

    other = threading.Thread(target=tick)
    was = gc.isenabled()
    gc.disable()   # as in analyze: a collection holds the lock too
    other.start()
    try:
        batch = patterns().ResultBatch(eng._tables, [doc] * n, rows, eng.max_events, 0.5, bytes(16 * n))
        t0 = time.perf_counter()
        batch.windows()
        t1 = time.perf_counter()
        assert len(batch.build_all(None, None, t0)) == n
        t2 = time.perf_counter()
    finally:
        stop.set()
        other.join()
        if was:
            gc.enable()
    for a, b in ((t0, t1), (t1, t2)):
        assert b - a < 0.02 or any(a + 0.3 * (b - a) < t < b - 0.3 * (b - a) for t in ticks)
