"""Pattern-match engine: batched pod logs -> AnalysisResult (replaces the
reference's log-parser REST hop, J/service/LogParserClient.java:36-55 /
LogParserRestClient.java:37-39).

GPU path (one call per batch of failures):
  host  : plan + pack logs into a pinned staging buffer (native, threaded)
  H2D   : one contiguous async copy
  device: ac_scan (DFA walk, LDS hot states) -> per-segment newline counts
          -> line_prefix (decoupled look-back exclusive prefix) -> scan_fixup
          (doc, factor, line, offset; newlines per doc), launched by one call
  D2H   : the (small) match list
  host  : factor -> matcher expansion, regex verification of candidate lines
          only, native event scoring (or the score_reduce kernel)
  device: context_spans: the +-k line window of every reported event, located in
          the text still resident from the scan (csrc/kernels/line_index.hip)
  host  : context lines decoded and result objects built natively
          (csrc/patterns/results.cpp)
The scan tail is eager: a captured hipGraph of it scanned a bucket-padded
length and cost more than the handful of launches it replaced (0.59 vs 0.40 ms per
64-log batch, profiles/scan_graph_vs_eager.jsonl); it was removed (docs/PARITY.md).
CPU path: the same post-processing fed by the pure-Python oracle.
"""
from __future__ import annotations

import bisect
import contextlib
import gc
import logging
import os
import threading
import time
import uuid
from collections.abc import Sequence
from dataclasses import dataclass

import numpy as np
import torch

from operator_amd.api.models import AnalysisEvent, AnalysisResult, AnalysisSummary, MatchedPattern
from operator_amd.patterns import oracle
from operator_amd.patterns.compiler import CompiledPatterns, compile_patterns
from operator_amd.patterns.schema import SEVERITIES, SEVERITY_RANK, PatternSet

log = logging.getLogger(__name__)

_EVENT_FIELDS = frozenset(AnalysisEvent.model_fields)
_SUMMARY_FIELDS = frozenset(AnalysisSummary.model_fields)
_RESULT_FIELDS = frozenset(AnalysisResult.model_fields)
_set_dict = object.__setattr__


def _mk(cls, d: dict, fields: frozenset):
    """A pydantic model from a COMPLETE dict of already-typed field values (the same
    object KModel.fast builds when every field is given: fields set = all of them, no
    extras), with the least Python per object."""
    m = cls.__new__(cls)
    _set_dict(m, "__dict__", d)
    _set_dict(m, "__pydantic_fields_set__", set(fields))
    _set_dict(m, "__pydantic_extra__", {})
    _set_dict(m, "__pydantic_private__", None)
    return m


@dataclass
class ScanStats:
    bytes_scanned: int = 0
    docs: int = 0
    raw_matches: int = 0
    verified_hits: int = 0
    scan_ms: float = 0.0
    host_ms: float = 0.0
    gpu_fallbacks: int = 0   # batches rescanned on the host after a GPU look-back timeout


class LazyResults(Sequence):
    """``MatchEngine.analyze(lazy=True)``: a batch's results, each built on first
    access and cached (a race builds one twice; the first stored copy wins)."""

    def __init__(self, build, n: int):
        self._build, self._items, self._lock = build, [None] * n, threading.Lock()

    def __len__(self) -> int:
        return len(self._items)

    def __getitem__(self, i):
        if isinstance(i, slice):
            return [self[j] for j in range(*i.indices(len(self._items)))]
        r = self._items[i]
        if r is None:
            r = self._build(i if i >= 0 else len(self._items) + i)
            with self._lock:
                if self._items[i] is None:
                    self._items[i] = r
                r = self._items[i]
        return r


@contextlib.contextmanager
def _gc_paused():
    """No cyclic-GC passes while a batch's results are allocated: each of the ~10^5 new
    objects of a 4096-log batch counts toward a collection, and the generation-2 passes
    they trigger re-scan every live object of the process (none of them a cycle)."""
    was = gc.isenabled()
    gc.disable()
    try:
        yield
    finally:
        if was:
            gc.enable()


def uuid4_strs(n: int) -> list[str]:
    """n random (version 4) UUID strings from one urandom call (uuid.uuid4() per result
    was a quarter of the host time of a 4096-result batch)."""
    raw = bytearray(os.urandom(16 * n))
    raw[6::16] = bytes((b & 0x0F) | 0x40 for b in raw[6::16])
    raw[8::16] = bytes((b & 0x3F) | 0x80 for b in raw[8::16])
    h = raw.hex()
    return [f"{h[i:i + 8]}-{h[i + 8:i + 12]}-{h[i + 12:i + 16]}-{h[i + 16:i + 20]}-{h[i + 20:i + 32]}"
            for i in range(0, 32 * n, 32)]


def _line_bounds(doc: bytes, off: int) -> tuple[int, int]:
    s = doc.rfind(b"\n", 0, off) + 1
    e = doc.find(b"\n", off)
    return s, (len(doc) if e < 0 else e)


def _context(doc: bytes, off: int, k: int) -> tuple[list[str], str]:
    s, e = _line_bounds(doc, off)
    line = doc[s:e]
    before = []
    ps = s
    for _ in range(k):
        if ps <= 0:
            break
        pe = ps - 1
        ps = doc.rfind(b"\n", 0, pe) + 1
        before.append(doc[ps:pe])
    after = []
    ne = e
    for _ in range(k):
        if ne >= len(doc):
            break
        ns = ne + 1
        if ns >= len(doc):
            break
        ne = doc.find(b"\n", ns)
        ne = len(doc) if ne < 0 else ne
        after.append(doc[ns:ne])
    ctx = [b.decode("utf-8", "replace") for b in reversed(before)] + [line.decode("utf-8", "replace")] + \
          [a.decode("utf-8", "replace") for a in after]
    return ctx, line.decode("utf-8", "replace")


def _line_offsets(doc: bytes) -> list[int]:
    offs = [0]
    i = doc.find(b"\n")
    while i >= 0:
        offs.append(i + 1)
        i = doc.find(b"\n", i + 1)
    return offs


class MatchEngine:
    """Compile a PatternSet once, then analyze batches of logs on one device."""

    SCAN_LANES = 256 * 1024   # ac_scan v2 streams on MI355X (256 CUs x 1024 threads)
    # hits that are scored natively, and whose results are built so: whole batches of 64 KiB logs with 2.6, 10, 41 and 82 thousand hits 3.4, 17, 89
    # and 189 ms, 6.9, 34, 162 and 339 by way of the GPU's sorts and Python's results; other threads wait no longer (results.cpp)
    HOST_SCORE_HITS = 1 << 16
    # context windows of a few logs' events are located on the host (3 events: 1 us against 30 for the round trip to the GPU);
    # larger batches leave the host to the next batch's packing
    HOST_CONTEXT_DOCS = 8
    HEAD_MATCHES = 2048       # match records read back with the count (a 64-log batch has some hundred)
    PACK_CHUNK = 16 << 20     # bytes of an upload while the host packs on (84 MB: 1.9 ms; 4 MB 2.0, 1 MB 2.5)
    PACK_FIRST = 2 << 20      # ... of the first one

    def __init__(self, patterns: PatternSet | CompiledPatterns, device: str | torch.device = "cuda",
                 seg_bytes: int = 1024, max_events: int = 50, significance: float = 0.5,
                 match_cap: int = 1 << 20, grid_blocks: int = 0, use_native_scorer: bool = True,
                 gpu_scorer: bool | None = None, profile_bytes: int = 1 << 20):
        self.cp = patterns if isinstance(patterns, CompiledPatterns) else compile_patterns(patterns)
        # DFA states are renumbered by visit count over the first `profile_bytes` of
        # text scanned (0: keep breadth-first numbering), see _profile_states
        self.profile_bytes = int(profile_bytes)
        self._profiled = False
        self.hot_coverage: tuple[float, float] | None = None
        self.device = torch.device(device)
        self.seg_bytes = int(seg_bytes)
        self.last_seg = self.seg_bytes   # segment size of the last scan (<= seg_bytes, see _scan_gpu)
        self.max_events = max_events
        self.significance = significance
        self.match_cap = int(match_cap)
        self.grid_blocks = grid_blocks
        self.pack_threads = max(1, min(16, (os.cpu_count() or 8)))
        self.use_native_scorer = use_native_scorer
        # score + rank events on the GPU (score.hip) when scanning there
        self.gpu_scorer = (self.device.type == "cuda") if gpu_scorer is None else gpu_scorer
        # ... unless it is asked for, only from HOST_SCORE_HITS hits on (the round trip to the GPU takes 65 us for 3 hits, 5 here)
        self._gpu_score_from = 0 if gpu_scorer else self.HOST_SCORE_HITS
        self._scorer = self._tables = None
        self._score_tables = None
        self.stats = ScanStats()
        # the scan's text and doc layout stay on the GPU until the next scan: the context
        # windows of the reported events are located there (line_index.hip context_spans)
        self._resident: tuple | None = None
        self._lock = threading.Lock()
        self._pinned: torch.Tensor | None = None
        self._text: torch.Tensor | None = None
        self._work: torch.Tensor | None = None
        self._head_h: torch.Tensor | None = None
        self._recs: torch.Tensor | None = None
        self._query_h: torch.Tensor | None = None
        self._span_h: torch.Tensor | None = None
        self._doc_newlines: tuple[list[bytes], list[int]] | None = None   # (docs, newlines) of the last GPU scan
        # matcher -> list of (pattern) where it is primary, for quick checks
        self._nm = self.cp.num_matchers
        fm_ptr = [0]
        fm_ids: list[int] = []
        for ms in self.cp.factor_matchers:
            fm_ids.extend(ms)
            fm_ptr.append(len(fm_ids))
        self._fm_ptr = np.asarray(fm_ptr, dtype=np.int64)
        self._fm_ids = np.asarray(fm_ids if fm_ids else [0], dtype=np.int64)
        self._verify = np.asarray(self.cp.matcher_verify + [False], dtype=bool)
        self._init_verifier()
        self._mp_cache: dict[int, MatchedPattern] = {}
        self._pinfo: list | None = None   # per-pattern (severity rank, MatchedPattern, remediation)
        self.last_timing: dict[str, float] = {}   # stage split of the last analyze() (host seconds)
        if self.device.type == "cuda" and self.cp.factors:
            self._upload_dfa()
        # Scans run on a stream of their own: the LLM engine keeps the default stream
        # busy with prefill/decode work, and a scan (and its result read-back) queued
        # behind that would wait for the whole queue before the prompt can be built.
        self._stream = torch.cuda.Stream(device=self.device) if self.device.type == "cuda" else None
        if self._stream is not None:
            torch.cuda.synchronize(self.device)   # DFA tables uploaded before the first scan

    def _init_verifier(self) -> None:
        """Per-matcher verification mode for the native post-processing (N4):
        0 = the factor hit is exact, 1 = native Pike-VM regex on the candidate line
        (patterns/nfa.py), 2 = Python ``re`` (outside the exactly-simulated subset)."""
        from operator_amd.ops import patterns
        from operator_amd.patterns.nfa import compile_nfa

        import re as _re

        progs, mode = [], []
        for i, m in enumerate(self.cp.matchers):
            if not self.cp.matcher_verify[i]:
                progs.append(None)
                mode.append(0)
                continue
            prog = compile_nfa(m.regex_source(), _re.IGNORECASE if m.ignore_case else 0)
            progs.append(prog)
            mode.append(1 if prog is not None else 2)
        self._mode = np.asarray(mode + [2], dtype=np.int8)
        self._rx = patterns().RegexSet(progs)
        self.native_verify = int(sum(1 for x in mode if x == 1))
        self.python_verify = int(sum(1 for x in mode if x == 2))

    def _on_stream(self):
        return torch.cuda.stream(self._stream) if self._stream is not None else contextlib.nullcontext()

    # ------------------------------------------------------------------ DFA upload
    def _upload_dfa(self) -> None:
        from operator_amd.ops import kernels

        d = self.cp.dfa
        dev = self.device
        S, log2c = int(d["num_states"]), int(d["log2_classes"])
        self.dfa_states, self.log2c = S, log2c
        self.cls_map = torch.frombuffer(bytearray(d["cls_map"]), dtype=torch.uint8).to(dev)
        self.table = torch.frombuffer(bytearray(d["table"]), dtype=torch.int16).reshape(S, 1 << log2c).to(dev)
        self.out_off = torch.frombuffer(bytearray(d["out_off"]), dtype=torch.int32).to(dev)
        self.out_ids = torch.frombuffer(bytearray(d["out_ids"]), dtype=torch.int32).to(dev)
        self.hot_states = int(min(S, kernels().max_hot_states(log2c)))
        self._build_hot_table(d["table"])

    def _build_hot_table(self, table: bytes) -> None:
        """ac_scan v2's LDS image: the first min(S, 256) states as full byte rows,
        [byte][state] with a 258-entry row stride (csrc/kernels/scan.h); and the per-state
        chain bytes its exact re-walk follows through cold states (patterns.cpp dfa_chain)."""
        from operator_amd.ops import kernels, patterns

        d = self.cp.dfa
        S, C = int(d["num_states"]), 1 << int(d["log2_classes"])
        stride = int(kernels().SCAN_HOT_STRIDE)
        H = min(S, stride - 2)
        tab = np.frombuffer(table, dtype=np.uint16).reshape(S, C)
        cls = np.frombuffer(d["cls_map"], dtype=np.uint8)
        wide = np.zeros((256, stride), dtype=np.uint16)
        wide[:, :H] = tab[:H][:, cls].T
        self.hot_table = torch.from_numpy(wide.view(np.int16).reshape(-1).copy()).to(self.device)
        chain = patterns().dfa_chain(table, int(d["log2_classes"]), S)
        self.chain = torch.frombuffer(bytearray(chain), dtype=torch.uint8).to(self.device)

    def _profile_states(self, sample: bytes) -> None:
        """Renumber DFA states by how often a walk over ``sample`` visits them, so the
        hot prefix ac_scan stages in LDS holds the states the logs actually sit in
        (breadth-first order leaves 42 % of wave byte-steps waiting on a global
        table read on the synthetic library; see csrc/patterns/patterns.cpp
        reorder_dfa). Match output does not depend on the numbering."""
        from operator_amd.ops import patterns

        d = self.cp.dfa
        r = patterns().reorder_dfa(d["table"], d["out_off"], d["out_ids"], int(d["log2_classes"]),
                                   int(d["num_states"]), d["cls_map"], sample, self.hot_states)
        dev = self.device
        S, C = int(d["num_states"]), 1 << int(d["log2_classes"])
        self.table = torch.frombuffer(bytearray(r["table"]), dtype=torch.int16).reshape(S, C).to(dev)
        self.out_off = torch.frombuffer(bytearray(r["out_off"]), dtype=torch.int32).to(dev)
        self.out_ids = torch.frombuffer(bytearray(r["out_ids"]), dtype=torch.int32).to(dev)
        self.hot_coverage = (float(r["hot_before"]), float(r["hot_after"]))
        self._build_hot_table(r["table"])
        self._profiled = True

    # ------------------------------------------------------------------ GPU scan
    def _ensure(self, name: str, numel: int, dtype, pinned: bool = False, device=None) -> torch.Tensor:
        t = getattr(self, name, None)
        if t is None or t.numel() < numel:
            cap = max(numel, int((t.numel() if t is not None else 0) * 1.5))
            if pinned:
                t = torch.empty(cap, dtype=dtype, pin_memory=True)
            else:
                t = torch.empty(cap, dtype=dtype, device=device or self.device)
            setattr(self, name, t)
        return t

    def scan_gpu(self, docs: list[bytes]) -> np.ndarray:
        """Raw factor hits as int64 array [n, 4] = (doc, factor, line, end_offset_in_doc)."""
        from operator_amd.utils.tracing import trace_range

        with trace_range(f"scan[{len(docs)}]"), self._on_stream():
            return self._scan_gpu(docs)

    def _scan_gpu(self, docs: list[bytes]) -> np.ndarray:
        hits, self._resident, self._doc_newlines = self._scan_gpu_slot(docs, 0)
        return hits

    def _scan_gpu_slot(self, docs: list[bytes], slot: int):
        """One scan in buffer set ``slot`` (0, or 1 for the second sub-batch in flight of a
        pipelined analyze). Returns (hits, resident, newlines): the text and layout the
        scan leaves on the GPU for the context windows, and (docs, newlines per doc);
        both None when the batch fell back to the host scan."""
        try:
            return self._scan_slot(docs, slot)
        except BaseException:
            # an upload may still be reading the pinned buffer, which the next scan writes into or replaces
            torch.cuda.current_stream(self.device).synchronize()
            raise

    def _scan_slot(self, docs: list[bytes], slot: int):
        from operator_amd.ops import kernels, patterns
        sfx = "" if slot == 0 else f"_s{slot}"

        P, C = patterns(), kernels()
        seg = self.seg_bytes
        # ac_scan v2 cuts the text into (CUs x 1024) equal streams of >= seg bytes: a
        # small batch (a 256-failure flagship wave is 16 MB) gets smaller segments so
        # that every CU has lanes to run
        approx = sum(len(d) + 1 for d in docs)
        while seg > 64 and approx // seg < self.SCAN_LANES:
            seg //= 2
        self.last_seg = seg
        lens = [len(d) for d in docs]
        total, first = P.plan_docs(lens, seg)
        n_segs, nd = total // seg, len(docs)
        # behind the text, in the same upload: first segment per doc (and the end), byte offset, length
        lay = 8 * (3 * nd + 1)
        pinned = self._ensure("_pinned" + sfx, total + lay, torch.uint8, pinned=True)
        text = self._ensure("_text" + sfx, total + lay, torch.uint8)
        layout = pinned[total:total + lay].numpy().view(np.int64)
        layout[:nd + 1] = first
        np.multiply(layout[:nd], seg, out=layout[nd + 1:2 * nd + 1])
        layout[2 * nd + 1:] = lens
        base_t, lens_t = text[total + 8 * (nd + 1):total + lay].view(torch.int64).split([nd, nd])
        # native threads pack the whole batch in order, and each doc-aligned chunk of >= PACK_CHUNK bytes is uploaded as soon
        # as it is in place, so a large batch pays max(pack, H2D) rather than the sum (a batch of 1.2 GB)
        threads = max(1, min(self.pack_threads, total >> 20))   # ~1 MB per packing thread (4.6 MB: 177 us on one, 93 on four)
        job = P.PackJob(docs, first, seg, pinned.data_ptr(), threads)
        try:
            a = 0
            while a < nd:
                chunk = self.PACK_CHUNK if a else self.PACK_FIRST
                b = min(nd, max(a + 1, bisect.bisect_left(first, first[a] + -(-chunk // seg), a + 1)))
                lo, hi = first[a] * seg, first[b] * seg
                job.wait(b)
                if self.profile_bytes > 0 and not self._profiled:
                    self._profile_states(pinned[:min(total, self.profile_bytes, hi)].numpy().tobytes())
                if b == nd:
                    hi += lay
                C.scan_upload(text, pinned, lo, hi)
                a = b
        finally:
            job.close()   # nothing writes into the buffer any more
        work = self._ensure("_work" + sfx, C.scan_work_bytes(n_segs), torch.uint8)
        # newlines per doc, the match count and an error word stand in front of the match records, and come back with the
        # first of those in one wait
        front = C.scan_report_bytes(nd)
        while True:
            recs = self._ensure("_recs" + sfx, front + 16 * self.match_cap, torch.uint8)
            cap = (recs.numel() - front) // 16
            head = min(self.HEAD_MATCHES, cap)
            host = self._ensure("_head_h" + sfx, front + 16 * head, torch.uint8, pinned=True)
            cnt, err = C.scan_batch(text, total, seg, nd, self.cls_map, self.table, self.log2c, self.hot_states, self.out_off,
                                    self.out_ids, self.hot_table, self.chain, self.grid_blocks, work, recs, cap, host, head)
            if err:
                # a line_prefix look-back hit its spin bound: the line numbers of this launch
                # are wrong, so the batch is recomputed on the host path instead
                log.warning("line_prefix look-back timed out; rescanning %d docs on the CPU path", nd)
                self.stats.gpu_fallbacks += 1
                return self.scan_cpu(docs), None, None
            if cnt <= cap:
                break
            self.match_cap = int(cnt * 1.25) + 1024  # overflow: grow and rescan (rare)
        self.stats.raw_matches += cnt
        self.stats.bytes_scanned += sum(lens)
        read = host.numpy()
        newlines = read[:8 * nd].view(np.int64).tolist()
        hits = read[front:front + 16 * cnt] if cnt <= head else recs[front:front + 16 * cnt].cpu().numpy()
        return hits.view(np.int32).reshape(-1, 4).astype(np.int64), (docs, base_t, lens_t, text), (docs, newlines)

    def _contexts_gpu(self, docs: list[bytes], queries: np.ndarray, resident: tuple | None = None, stream=None) -> np.ndarray | None:
        """(window start, window end, line start, line end) of every query (doc, byte offset, lines), located in the text the last GPU
        scan (or the given ``resident`` one) left on the GPU; None when that scan was not of ``docs``: the host path."""
        from operator_amd.ops import kernels

        r = self._resident if resident is None else resident
        if r is None or r[0] is not docs or not len(queries):
            return None
        _, base, lens, text = r
        n = len(queries)
        q, out = self._ensure("_query_h", 3 * n, torch.int64, pinned=True), self._ensure("_span_h", 4 * n, torch.int64, pinned=True)
        q.numpy()[:3 * n] = queries.reshape(-1)
        # the kernel runs on the scan stream, behind the scan, and reads and writes pinned memory: no copy on a stream that the
        # LLM's decode graphs keep busy for tens of ms
        with (torch.cuda.stream(stream) if stream is not None else self._on_stream()):
            kernels().context_spans(text, base, lens, q, out, n)
        return out.numpy()[:4 * n].reshape(n, 4)

    def scan_cpu(self, docs: list[bytes]) -> np.ndarray:
        """Same contract as scan_gpu, computed with Python (used without a GPU)."""
        rows = []
        lows = [f for f in self.cp.factors]
        for di, d in enumerate(docs):
            dl = d.lower()
            for fi, f in enumerate(lows):
                start = 0
                while True:
                    i = dl.find(f, start)
                    if i < 0:
                        break
                    end = i + len(f) - 1
                    line = dl.count(b"\n", 0, end)
                    rows.append((di, fi, line, end))
                    start = i + 1
        return np.asarray(rows, dtype=np.int64).reshape(-1, 4)

    # ------------------------------------------------------------------ analysis
    def hits(self, docs: list[bytes]) -> tuple[np.ndarray, dict]:
        """Verified, de-duplicated matcher hits [n, 3] = (doc, matcher, line) + offsets."""
        return self._split_hits(self._scan_and_verify(docs))

    @staticmethod
    def _split_hits(rows: np.ndarray) -> tuple[np.ndarray, dict]:
        return np.ascontiguousarray(rows[:, :3]), dict(zip(map(tuple, rows[:, :3].tolist()), rows[:, 3].tolist()))

    def _scan_and_verify(self, docs: list[bytes]) -> np.ndarray:
        t0 = time.perf_counter()
        raw = self.scan_gpu(docs) if (self.device.type == "cuda" and self.cp.factors) else (
            self.scan_cpu(docs) if self.cp.factors else np.zeros((0, 4), np.int64))
        return self._verified(docs, raw, t0)

    def _verified(self, docs: list[bytes], raw: np.ndarray, t0: float) -> np.ndarray:
        """Hits [n, 4] = (doc, matcher, line, byte offset), each (doc, matcher, line) once, in order."""
        t1 = time.perf_counter()
        from operator_amd.ops import patterns

        P = patterns()
        # native: factor -> matcher expansion, candidate-line verification (Pike VM),
        # (doc, matcher, line) de-duplication; Python `re` only for matchers outside
        # the NFA subset (`pending`)
        done, pending = P.postprocess_hits(raw.reshape(-1, 4), self._fm_ptr, self._fm_ids, self._mode, docs, self._rx)
        parts = [done]
        if pending.shape[0]:
            keep = []
            for d_, m_, l_, o_ in pending.tolist():
                s_, e_ = _line_bounds(docs[d_], o_)
                if self.cp.regexes[m_].search(docs[d_][s_:e_]) is not None:
                    keep.append((d_, m_, l_, o_))
            parts.append(np.asarray(keep, dtype=np.int64).reshape(-1, 4))
        # matchers with no usable factor: evaluated on every line on the CPU
        for m_ in self.cp.unfiltered:
            if self._rx.has(m_):
                parts.append(P.line_scan(docs, self._rx, m_))
                continue
            rx = self.cp.regexes[m_]
            rows = []
            for d_, doc_b in enumerate(docs):
                lo = _line_offsets(doc_b)
                for li, ls in enumerate(lo):
                    le = lo[li + 1] - 1 if li + 1 < len(lo) else len(doc_b)
                    if rx.search(doc_b[ls:le]):
                        rows.append((d_, m_, li, max(ls, le - 1) if le > ls else ls))
            parts.append(np.asarray(rows, dtype=np.int64).reshape(-1, 4))
        allh = np.concatenate(parts, 0) if len(parts) > 1 else done
        if len(parts) > 1 and allh.shape[0]:
            order = np.lexsort((allh[:, 2], allh[:, 1], allh[:, 0]))
            allh = allh[order]
            keep = np.ones(allh.shape[0], dtype=bool)
            keep[1:] = np.any(allh[1:, :3] != allh[:-1, :3], axis=1)
            allh = allh[keep]
        self.stats.verified_hits += allh.shape[0]
        self.stats.scan_ms += (t1 - t0) * 1e3
        self.stats.host_ms += (time.perf_counter() - t1) * 1e3
        return allh

    def _gpu_tables(self):
        """Static pattern tables for score.hip (CSR), uploaded once per pattern set."""
        if self._score_tables is None:
            cp, dev = self.cp, self.device
            pats = cp.patset.patterns
            nm = cp.num_matchers
            prim_of: list[list[int]] = [[] for _ in range(nm)]
            for p_, m_ in enumerate(cp.pattern_primary):
                prim_of[m_].append(p_)
            prim_ptr = np.zeros(nm + 1, np.int64)
            prim_ptr[1:] = np.cumsum([len(x) for x in prim_of])
            sec_ptr = np.zeros(len(pats) + 1, np.int64)
            sec_ptr[1:] = np.cumsum([len(p.secondary) for p in pats])
            t = lambda a, dt=torch.int32: torch.as_tensor(np.asarray(a), dtype=dt).to(dev)  # noqa: E731
            self._score_tables = dict(
                npat=np.asarray([len(x) for x in prim_of], np.int64),
                prim_ptr=t(prim_ptr), prim_pat=t([p_ for x in prim_of for p_ in x] or [0]),
                sec_ptr=t(sec_ptr), sec_matcher=t([m_ for x in cp.pattern_secondary for m_ in x] or [0]),
                sec_w=t([s_.weight for p in pats for s_ in p.secondary] or [0.0], torch.float64),
                sec_win=t([s_.window for p in pats for s_ in p.secondary] or [0]),
                conf=t([p.primary.confidence for p in pats], torch.float64),
                severity=t([p.severity_rank for p in pats]), severity_h=[p.severity_rank for p in pats])
        return self._score_tables

    def _events_gpu(self, hits: np.ndarray, n_docs: int) -> list[list[oracle.Event]]:
        from operator_amd.ops import kernels

        T = self._gpu_tables()
        dev = self.device
        n = hits.shape[0]
        doc, mat, line = hits[:, 0], hits[:, 1], hits[:, 2]
        doc_ptr = np.zeros(n_docs + 1, np.int64)
        doc_ptr[1:] = np.cumsum(np.bincount(doc, minlength=n_docs))
        nm = T["npat"].shape[0]
        per_hit = np.where(mat < nm, T["npat"][np.minimum(mat, nm - 1)], 0)
        ev_ptr = np.zeros(n + 1, np.int64)
        ev_ptr[1:] = np.cumsum(per_hit)
        ev_doc_ptr = ev_ptr[doc_ptr]
        E = int(ev_ptr[-1])
        # one upload (keys, then the int32 index arrays) and one read-back (scores, then the int32 columns)
        parts = (doc, doc_ptr, ev_ptr, ev_doc_ptr)
        buf = torch.empty(8 * n + 4 * sum(map(len, parts)), dtype=torch.uint8, pin_memory=True)
        host = buf.numpy()
        np.bitwise_or(mat << 32, line, out=host[:8 * n].view(np.int64))
        np.concatenate(parts, out=host[8 * n:].view(np.int32), casting="same_kind")
        buf = buf.to(dev, non_blocking=True)
        keys, ints = buf[:8 * n].view(torch.int64), buf[8 * n:].view(torch.int32).split([len(x) for x in parts])
        res = torch.empty(20 * E, dtype=torch.uint8, device=dev)
        ev_score, (ev_pat, ev_line, order) = res[:8 * E].view(torch.float64), res[8 * E:].view(torch.int32).split([E] * 3)
        summary = torch.empty(3 * max(n_docs, 1), dtype=torch.int32, device=dev)
        kernels().score_events(keys, ints[0], ints[1], T["prim_ptr"], T["prim_pat"], ints[2], ints[3], T["sec_ptr"], T["sec_matcher"],
                               T["sec_w"], T["sec_win"], T["conf"], T["severity"], float(self.significance), ev_score, ev_pat, ev_line,
                               order, summary)
        res = res.cpu().numpy()
        sc, (pt, ln, od) = res[:8 * E].view(np.float64), res[8 * E:].view(np.int32).reshape(3, E)
        sev = T["severity_h"]
        out = []
        for d in range(n_docs):
            a, b = int(ev_doc_ptr[d]), int(ev_doc_ptr[d + 1])
            if b - a > 2048:  # beyond the LDS sort cap: rank on the host (same key)
                idx = sorted(range(a, b), key=lambda i: (-sc[i], -sev[pt[i]], ln[i], pt[i]))
            else:
                idx = od[a:b]
            out.append([oracle.Event(int(pt[i]), int(ln[i]), float(sc[i])) for i in idx])
        return out

    def events(self, docs: list[bytes]) -> tuple[list[list[oracle.Event]], dict]:
        hits, offs = self.hits(docs)
        return self._events_from_hits(docs, hits), offs

    def _scores_on_gpu(self, hits: int) -> bool:
        return self.gpu_scorer and self.device.type == "cuda" and not (self.use_native_scorer and hits <= self._gpu_score_from)

    def _native_scorer(self):
        if self._scorer is None:   # the pattern tables, once per engine
            from operator_amd.ops import patterns

            cp, pats = self.cp, self.cp.patset.patterns
            self._scorer = patterns().Scorer(
                cp.pattern_primary, [p.primary.confidence for p in pats], [p.severity_rank for p in pats],
                cp.pattern_secondary, [[s.weight for s in p.secondary] for p in pats],
                [[s.window for s in p.secondary] for p in pats], cp.num_matchers)
        return self._scorer

    def _events_from_hits(self, docs: list[bytes], hits: np.ndarray, stream=None) -> list[list[oracle.Event]]:
        cp = self.cp
        if self._scores_on_gpu(len(hits)):
            with (torch.cuda.stream(stream) if stream is not None else self._on_stream()):
                return self._events_gpu(hits, len(docs))
        if self.use_native_scorer:
            evs = [[oracle.Event(*e) for e in d] for d in self._native_scorer().score(hits, len(docs))]
        else:
            per: list[set] = [set() for _ in docs]
            for d_, m_, l_ in hits.tolist():
                per[d_].add((m_, l_))
            evs = [oracle.score_doc(cp, h) for h in per]
        return evs

    def analyze(self, docs: list[bytes], pods: list[tuple[str, str]] | None = None,
                lazy: bool = False) -> "list[AnalysisResult] | LazyResults":
        """Full AnalysisResult per doc (pods = [(name, namespace)] for labelling).

        ``lazy``: return once the batch's per-doc event lists and their context windows
        exist (scan, verify, score, one batched context call); each doc's result objects
        are built on first access (``LazyResults``) — the consumer that reads result i
        pays for it (~10 us), and the scan engine is free for the next batch that much
        sooner."""
        with self._lock, _gc_paused():
            t0 = time.perf_counter()
            subs = self._sub_batches(docs)
            if subs is not None:
                return self._analyze_pipelined(docs, pods, lazy, subs, t0)
            self._doc_newlines = None
            score = self._score(docs, self._scan_and_verify(docs))
            t_ev = time.perf_counter()
            nls = self._doc_newlines[1] if self._doc_newlines and self._doc_newlines[0] is docs else None
            self._doc_newlines = None
            self.stats.docs += len(docs)
            build, build_all = self._finish(docs, score, nls, None, None, pods, t0)
            t_ctx = time.perf_counter()
            if lazy:
                # contexts are done (one batched call); only the result objects are
                # deferred to their first access
                self.last_timing = {"events_s": t_ev - t0, "contexts_s": t_ctx - t_ev}
                ms = (t_ctx - t0) * 1e3
                return LazyResults(lambda di: build(di, ms), len(docs))
            out = build_all()
            t_end = time.perf_counter()
            self.last_timing = {"events_s": t_ev - t0, "contexts_s": t_ctx - t_ev, "results_s": t_end - t_ctx}
            return out

    # ------------------------------------------------------------------ pipelined analyze
    PIPE_MIN_BYTES = 192 << 20   # batches at least this large are analysed in sub-batches
    PIPE_SUB_BYTES = 160 << 20   # bytes per sub-batch (doc-aligned)

    def _sub_batches(self, docs: list[bytes]) -> list[tuple[int, int]] | None:
        """Doc-aligned (lo, hi) sub-batches of about PIPE_SUB_BYTES for a large GPU batch,
        else None. A batch of 1.2 GB is H2D-bound on the GPU (~24 ms of its
        ~27 ms scan) and host-bound after it (~60 ms of verification, scoring, context
        windows and result objects): in sub-batches the next one's pack + H2D + scan runs
        while the host finishes the previous one."""
        if self.device.type != "cuda" or not self.cp.factors or self.PIPE_SUB_BYTES <= 0 or len(docs) < 2:
            return None
        total = sum(map(len, docs))
        if total < self.PIPE_MIN_BYTES:
            return None
        n = min(len(docs), max(2, -(-total // self.PIPE_SUB_BYTES)))
        bounds, acc, k = [0], 0, 1
        for i, d in enumerate(docs[:-1]):
            acc += len(d)
            if acc * n >= total * k:
                bounds.append(i + 1)
                k += 1
        bounds.append(len(docs))
        return [(lo, hi) for lo, hi in zip(bounds, bounds[1:]) if hi > lo]

    def _analyze_pipelined(self, docs: list[bytes], pods, lazy: bool, subs: list[tuple[int, int]], t0: float):
        """analyze() over sub-batches: a worker thread scans sub-batch i + 1 (pack, H2D,
        ac_scan, line index, match read-back; buffer set i % 2, on the scan stream) while
        this thread verifies, scores and builds sub-batch i (GPU scoring and context
        windows on a second stream, so they do not queue behind the next scan's copies).
        A buffer set is rescanned only after its context windows were read (``free``)."""
        import queue

        if getattr(self, "_stream2", None) is None:
            self._stream2 = torch.cuda.Stream(device=self.device)
        ready: queue.Queue = queue.Queue()
        free = threading.Semaphore(2)
        stop = threading.Event()

        def worker():
            try:
                for i, (lo, hi) in enumerate(subs):
                    free.acquire()
                    if stop.is_set():
                        return
                    sub = docs[lo:hi]
                    with self._on_stream():
                        ready.put((i, sub) + self._scan_gpu_slot(sub, i % 2) + (time.perf_counter(),))
            except BaseException as e:   # noqa: BLE001 -- re-raised on the analysing thread
                ready.put(e)

        th = threading.Thread(target=worker, name="oamd-scan-pipe", daemon=True)
        th.start()
        builds: list = []
        t_host = t_ctx_total = 0.0
        try:
            for _ in subs:
                item = ready.get()
                if isinstance(item, BaseException):
                    raise item
                i, sub, raw, resident, nl, _ = item
                u0 = time.perf_counter()
                score = self._score(sub, self._verified(sub, raw, u0), self._stream2)
                u1 = time.perf_counter()
                nls = nl[1] if nl is not None and nl[0] is sub else None
                lo = subs[i][0]
                build = self._finish(sub, score, nls, resident, self._stream2, pods[lo:subs[i][1]] if pods else None, t0)
                free.release()   # this buffer set's text is no longer needed
                u2 = time.perf_counter()
                t_host += u1 - u0
                t_ctx_total += u2 - u1
                builds.append((lo, subs[i][1], *build))
        finally:
            stop.set()
            free.release()
            free.release()
            th.join()
        self._resident = None
        self._doc_newlines = None
        self.stats.docs += len(docs)
        t_ctx = time.perf_counter()
        owner = [0] * len(docs)
        for bi, (lo, hi, *_) in enumerate(builds):
            owner[lo:hi] = [bi] * (hi - lo)
        if lazy:
            ms = (t_ctx - t0) * 1e3
            self.last_timing = {"subs": len(subs), "events_s": t_host, "contexts_s": t_ctx_total,
                                "pipelined_s": t_ctx - t0}

            def get(di: int):
                lo, _, build, _ = builds[owner[di]]
                return build(di - lo, ms)

            return LazyResults(get, len(docs))
        out = []
        for _, _, _, build_all in builds:
            out.extend(build_all())
        t_end = time.perf_counter()
        self.last_timing = {"subs": len(subs), "events_s": t_host, "contexts_s": t_ctx_total,
                            "results_s": t_end - t_ctx, "pipelined_s": t_ctx - t0}
        return out

    def _score(self, docs: list[bytes], rows: np.ndarray, stream=None):
        """The events of verified hits: a native batch (csrc/patterns/results.cpp), which goes on to the results by itself, or, scored
        on the GPU or in Python, (events per doc, byte offset by (doc, matcher, line))."""
        if not self.use_native_scorer or self._scores_on_gpu(len(rows)):
            hits, offs = self._split_hits(rows)
            return self._events_from_hits(docs, hits, stream), offs
        from operator_amd.ops import patterns

        if self._tables is None:
            info, pats = self._pattern_info(), self.cp.patset.patterns
            self._tables = patterns().ResultTables(
                self._native_scorer(), [p.context_lines for p in pats], [r for r, _, _ in info], [mp for _, mp, _ in info],
                [rem for _, _, rem in info], SEVERITIES, AnalysisEvent, _EVENT_FIELDS, AnalysisSummary, _SUMMARY_FIELDS,
                AnalysisResult, _RESULT_FIELDS, self._engine_name())
        return patterns().ResultBatch(self._tables, docs if type(docs) is list else list(docs), rows, self.max_events, self.significance,
                                      os.urandom(16 * len(docs)))

    def _finish(self, docs: list[bytes], score, nls, resident, stream, pods, t0: float):
        """The context windows of every reported event of ``docs`` (one batched call), then ``build(i, ms)`` for result i and
        ``build_all()``, whose processing times are measured as they are built."""
        from operator_amd.ops import patterns

        on_gpu = len(docs) > self.HOST_CONTEXT_DOCS
        if not isinstance(score, tuple):
            spans = self._contexts_gpu(docs, score.queries(), resident, stream) if on_gpu and len(score) else None
            score.windows(spans)

            def build(di: int, ms: float) -> AnalysisResult:
                pod = pods[di] if pods else (None, None)
                return score.build(di, pod[0], pod[1], -1 if nls is None else nls[di], ms)

            return build, lambda: score.build_all(pods or None, nls, t0)
        evs, offs = score
        ids = uuid4_strs(len(docs))
        # the +-k context windows of every reported event, extracted natively in one
        # call over the whole batch (N3)
        q_doc, q_off, q_k = [], [], []
        for di, (doc, ev) in enumerate(zip(docs, evs)):
            o_, k_ = self._context_queries(di, doc, ev, offs)
            q_doc.extend([di] * len(o_))
            q_off.extend(o_)
            q_k.extend(k_)
        ctxs = []
        if q_doc:
            spans = self._contexts_gpu(docs, np.stack([q_doc, q_off, q_k], 1), resident, stream) if on_gpu else None
            P = patterns()
            ctxs = P.contexts(docs, q_doc, q_off, q_k) if spans is None else P.contexts_from_spans(docs, q_doc, spans)
        starts = [0]
        for ev in evs:
            starts.append(starts[-1] + min(len(ev), self.max_events))

        def build_one(di: int, ms: float | None = None) -> AnalysisResult:
            return self._result(docs[di], evs[di], ctxs[starts[di]:starts[di + 1]],
                                pods[di] if pods else (None, None),
                                (time.perf_counter() - t0) * 1e3 if ms is None else ms,
                                None if nls is None else nls[di], ids[di])

        return build_one, lambda: [build_one(di) for di in range(len(docs))]

    def _context_queries(self, di: int, doc: bytes, ev: list[oracle.Event], offs: dict) -> tuple[list, list]:
        """(byte offset, context lines) of each reported event of doc ``di``: the offset
        of its primary matcher's hit on that line (the line start if none is known)."""
        cp = self.cp
        pats = cp.patset.patterns
        q_off, q_k = [], []
        lo = None
        for e in ev[: self.max_events]:
            off = offs.get((di, cp.pattern_primary[e.pattern], e.line))
            if off is None:
                if lo is None:
                    lo = _line_offsets(doc)
                off = lo[e.line] if e.line < len(lo) else 0
            q_off.append(off)
            q_k.append(pats[e.pattern].context_lines)
        return q_off, q_k

    def _engine_name(self) -> str:
        return "gpu-ac" if self.device.type == "cuda" else "cpu-oracle"

    def _matched(self, pi: int) -> MatchedPattern:
        mp = self._mp_cache.get(pi)
        if mp is None:   # immutable per pattern: built once, shared by every event
            p = self.cp.patset.patterns[pi]
            mp = self._mp_cache[pi] = MatchedPattern.fast(
                id=p.id, name=p.name, severity=p.severity, category=p.category or None, library=p.library or None)
        return mp

    def _pattern_info(self) -> list:
        """Per pattern, built once: (severity rank, MatchedPattern, remediation or None)."""
        if self._pinfo is None:
            self._pinfo = [(p.severity_rank, self._matched(i), p.remediation or None)
                           for i, p in enumerate(self.cp.patset.patterns)]
        return self._pinfo

    def _result(self, doc: bytes, ev: list[oracle.Event], ctxs: list, pod, ms: float,
                newlines: int | None = None, analysis_id: str | None = None) -> AnalysisResult:
        # the hot host loop of a scan batch (4096 results of 290 KiB logs): per-pattern
        # constants looked up once (_pattern_info), severities counted by rank, and every
        # model built by _mk from a complete field dict (all fields given, so no defaults /
        # factories to merge)
        info = self._pattern_info()
        counts = [0, 0, 0, 0, 0]
        sig = 0
        hi = -1
        thr = self.significance
        for e in ev:
            r = info[e.pattern][0]
            counts[r] += 1
            if r > hi:
                hi = r
            if e.score >= thr:
                sig += 1
        events = []
        for e, (ctx, line) in zip(ev[: self.max_events], ctxs):
            _, mp, rem = info[e.pattern]
            events.append(_mk(AnalysisEvent, {"line_number": e.line + 1, "matched_pattern": mp,
                                              "score": round(e.score, 6), "context": ctx, "matched_line": line,
                                              "remediation": rem}, _EVENT_FIELDS))
        summary = _mk(AnalysisSummary, {"highest_severity": SEVERITIES[hi] if hi >= 0 else None,
                                        "significant_events": sig, "total_events": len(ev),
                                        "severity_distribution": {SEVERITIES[i]: c for i, c in enumerate(counts) if c}},
                      _SUMMARY_FIELDS)
        return _mk(AnalysisResult, {
            "analysis_id": analysis_id or str(uuid.uuid4()), "pod_name": pod[0], "pod_namespace": pod[1],
            "events": events, "summary": summary,
            "metadata": {"engine": self._engine_name(),
                         "patternsChecked": len(info),
                         "totalLines": (doc.count(b"\n") if newlines is None else newlines) + 1,
                         "bytes": len(doc), "processingTimeMs": round(ms, 3)}}, _RESULT_FIELDS)
