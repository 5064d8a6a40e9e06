"""Performance cases: what users have this framework do, from one call to a full batch.

Four kinds of work, each through the entry point a program calls:

scan     pod logs against a pattern library, host bytes in, analysis results out
         (``MatchEngine.analyze``; the operator's pattern stage and the log-parser endpoint).
prefill  new prompts through a served model as one packed batch, the logits that pick each
         prompt's first token out (``LLMEngine.given_start``).
decode   one token further for a batch of running sequences, their logits out
         (``LLMEngine.given_next`` on the captured decode graphs).
experts  a routed feed-forward of the expert design with the routes given, up to the next sublayer's
         input (``ops.decoder.experts`` and ``stream_step``). On its own, because behind a router of
         random weights a token between two experts takes either one, whatever the precision.

Models are the presets of ``models/config.py`` at their full width, heads and vocabulary, cut to
a few layers (as ``bench.py --model-speed`` does) so that a pass stays short; weights are random
(``init_random``), prompts uniform random tokens. Lengths follow the operator's explanations:
prompts of 885 tokens (at most 1024), answers of up to 500, batches of up to 256, logs of 64 KiB
in batches of up to 64 against 1000 patterns, 290 KiB logs for bulk scans.
"""
from __future__ import annotations

import functools
import hashlib
import math
import random
import re
from dataclasses import replace

import numpy as np
import torch

from operator_amd import ops
from operator_amd.engine.llm import LLMEngine
from operator_amd.engine.match import MatchEngine
from operator_amd.models.config import LatentSpec, get_config
from operator_amd.models.kv_cache import PagedKVCache
from operator_amd.models.registry import build_model
from operator_amd.ops import decoder as dec
from operator_amd.patterns.compiler import compile_patterns
from operator_amd.patterns.synth import LogFactory, synthetic_library

PAGE = 16   # tokens of a cache page
SAME_WEIGHTS = 1   # every prepared model holds these weights; a case's seed makes its tokens and logs


def _scan(name: str | None, docs: int, kib: int, patterns: int = 1000) -> dict:
    return _named(name, {"kind": "scan", "docs": docs, "kib": kib, "patterns": patterns})


def _model(name: str | None, kind: str, model: str, seqs: int, tokens: int, spread: float = 0.0, layers: int = 4,
           dtype: str = "bfloat16", weights: str = "bfloat16") -> dict:
    """``seqs`` sequences of ``tokens`` tokens, give or take the share ``spread`` of them."""
    return _named(name, {"kind": kind, "model": model, "seqs": seqs, "tokens": tokens, "spread": spread, "layers": layers,
                         "dtype": dtype, "weights": weights})


def _experts(name: str | None, model: str, tokens: int) -> dict:
    return _named(name, {"kind": "experts", "model": model, "tokens": tokens})


def _named(name: str | None, case: dict) -> dict:
    return case if name is None else {"name": name, **case}


def listed() -> list[dict]:
    return [
        # one failed pod: its log on its own, nothing to batch it with
        _scan("scan-one", 1, 64),
        # a failure wave: the scan service's largest batch of 64 KiB logs
        _scan("scan-wave", 64, 64),
        # a backlog of whole log files handed over at once
        _scan("scan-bulk", 256, 290),
        # one failed pod: its explanation prompt, alone, on the default model
        _model("prefill-one", "prefill", "llama3-8b", 1, 885),
        # a wave of failures: a full prefill batch of explanation prompts
        _model("prefill-wave", "prefill", "llama3-8b", 32, 885, 0.15),
        # one explanation being written
        _model("decode-one", "decode", "llama3-8b", 1, 1130),
        # a full batch of explanations being written, prompts and answers at every length
        _model("decode-wave", "decode", "llama3-8b", 256, 1150, 0.3),
        # the large model with fp8 weights, a quarter-full batch
        _model("decode-fp8", "decode", "llama3-70b", 64, 1100, 0.2, layers=2, weights="fp8"),
        # the expert design's routed layer: some prompts at once, and a small odd batch being written
        _experts("experts-prompts", "sufolix-8b", 7950),
        _experts("experts-batch", "sufolix-8b", 21),
        # the window / latent attention design on long contexts
        _model("decode-latent", "decode", "relurax-8b", 48, 3600, 0.1),
        # a small model of that design in fp32 (trace replay, reference logits)
        _model("prefill-f32", "prefill", "relurax-1b", 2, 500, 0.1, dtype="float32"),
    ]


# models of the drawn cases: layers (of the expert design those without a router), dtype, weights
DRAWN = (("llama3-8b", 4, "bfloat16", "bfloat16"), ("mistral-7b", 4, "bfloat16", "bfloat16"), ("qwen2.5-7b", 4, "bfloat16", "bfloat16"),
         ("llama-1b-hd128", 4, "bfloat16", "bfloat16"), ("llama3-70b", 2, "bfloat16", "fp8"), ("llama3-8b", 4, "bfloat16", "fp8"),
         ("sufolix-8b", 1, "bfloat16", "bfloat16"), ("sufolix-1b", 1, "bfloat16", "bfloat16"), ("relurax-8b", 4, "bfloat16", "bfloat16"),
         ("relurax-1b", 4, "bfloat16", "bfloat16"), ("sufolix-1b", 1, "float32", "bfloat16"), ("relurax-1b", 4, "float32", "bfloat16"))


def _log_size(rng: random.Random, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(("scan", "prefill", "prefill", "prefill", "decode", "decode", "decode", "experts"))
    if kind == "experts":
        return _experts(None, rng.choice(("sufolix-8b", "sufolix-1b")), _log_size(rng, 1, 8192))
    if kind == "scan":
        kib = _log_size(rng, 4, 512)
        return _scan(None, min(_log_size(rng, 1, 256), 256 * 290 // kib), kib, rng.choice((25, 200, 1000)))
    model, layers, dtype, weights = rng.choice(DRAWN)
    spread = round(rng.uniform(0.0, 0.4), 2)
    if kind == "prefill":
        tokens = _log_size(rng, 24, 2048)
        total = 2048 if dtype == "float32" else 16384 if model == "llama3-70b" else 28320
        seqs = min(_log_size(rng, 1, 32), max(1, total // tokens))
    else:
        tokens = _log_size(rng, 96, 4096)
        seqs = min(_log_size(rng, 1, 32 if dtype == "float32" else 256), max(1, (32768 if dtype == "float32" else 196608) // tokens))
    return _model(None, kind, model, seqs, tokens, spread, layers, dtype, weights)


# ---------------------------------------------------------------- what a case consists of
def _config(case: dict):
    cfg = get_config(case["model"])
    if hasattr(cfg, "layer_specs"):
        return replace(cfg, layer_specs=cfg.layer_specs[:case["layers"]])
    return replace(cfg, layers=case["layers"])


def _lengths(case: dict) -> list[int]:
    """Tokens of every sequence: spread evenly over the case's range, in no order."""
    n, m, s = case["seqs"], case["tokens"], case["spread"]
    return [max(2, round(m * (1 + s * (2 * ((i * 0.6180339887 + 0.5) % 1.0) - 1)))) for i in range(n)]


def _tokens(case: dict, seed: int) -> list[list[int]]:
    rng = np.random.default_rng([seed, 7])
    vocab = get_config(case["model"]).vocab_size
    return [rng.integers(0, vocab, n).tolist() for n in _lengths(case)]


def _logs(case: dict, seed: int) -> list[bytes]:
    return LogFactory(case["patterns"], seed=seed % (1 << 31), pool_lines=4096).batch(case["docs"], case["kib"] * 1024)[0]


@functools.lru_cache(maxsize=4)
def _library(patterns: int):
    return compile_patterns(synthetic_library(patterns, seed=0))


def prepare(case: dict, seed: int) -> dict:
    if case["kind"] == "scan":
        compiled = _library(case["patterns"])
        return {"kind": "scan", "engine": MatchEngine(compiled, device="cuda"), "docs": _logs(case, seed),
                "index": {p.id: i for i, p in enumerate(compiled.patset.patterns)}}
    if case["kind"] == "experts":
        return _prepare_experts(case, seed)
    cfg, lens = _config(case), _lengths(case)
    dtype = getattr(torch, case["dtype"])
    model = build_model(cfg, device="cuda", dtype=dtype, weight_dtype=case["weights"]).init_random(SAME_WEIGHTS)
    kv = PagedKVCache.for_model(model, sum(n // PAGE + 2 for n in lens), PAGE)
    eng = LLMEngine(model, kv, max_batch=256, max_context=8192, prefill_graphs=False, prefix_sharing=False)
    st = {"kind": case["kind"], "engine": eng, "prompts": _tokens(case, seed)}
    if case["kind"] == "decode":
        # every sequence but its last token is in the cache; a pass gives that one
        st["next"] = [p.pop() for p in st["prompts"]]
        st["reqs"] = []
        for a in range(0, len(lens), 8):
            st["reqs"] += eng.given_start(st["prompts"][a:a + 8], [[]] * len(lens[a:a + 8]))[0]
        bucket = next(b for b in eng.buckets if b >= min(len(lens), eng.max_batch))
        eng.warmup([bucket])
    else:
        st["want"] = [[len(p) - 1] for p in st["prompts"]]
    return st


def _expert_layer(case: dict):
    """(configuration, its routed feed-forward, raw weights by name)."""
    cfg = get_config(case["model"])
    f = cfg.layer_specs[1].mlp
    w = _Weights(torch.bfloat16)
    raw = {n: [w(f"e{e}.{n}", shape, 1.0 / math.sqrt(shape[1])) for e in range(f.experts)]
           for n, shape in (("gate", (f.ff, cfg.hidden)), ("up", (f.ff, cfg.hidden)), ("down", (cfg.hidden, f.ff)))}
    return cfg, f, raw


def _expert_inputs(case: dict, cfg, f, seed: int) -> dict:
    """Normalised tokens, their routes (some experts are asked for more than others) and the streams."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    T, E, S = case["tokens"], f.experts, cfg.streams
    score = torch.randn(T, E, generator=g, device="cuda") + 0.5 * torch.randn(E, generator=g, device="cuda")
    wt, ids = torch.sigmoid(score).topk(f.top, -1)
    return {"h": torch.randn(T, cfg.hidden, generator=g, device="cuda").bfloat16(), "ids": ids.int(), "wt": wt.contiguous(),
            "x": torch.randn(T, S, cfg.hidden, generator=g, device="cuda"),
            "mix": torch.eye(S, device="cuda") + 0.05 * torch.randn(S, S, generator=g, device="cuda"),
            "out": 1.0 + 0.1 * torch.randn(S, generator=g, device="cuda"),
            "inp": 1.0 / S + 0.1 * torch.randn(S, generator=g, device="cuda"),
            "norm": 1.0 + 0.1 * torch.randn(cfg.hidden, generator=g, device="cuda")}


def _prepare_experts(case: dict, seed: int) -> dict:
    cfg, f, raw = _expert_layer(case)
    return {"kind": "experts", "cfg": cfg, "top": f.top, "wd": torch.stack(raw["down"]),
            "wgu": torch.stack([ops.interleave_gate_up(g, u) for g, u in zip(raw["gate"], raw["up"])]),
            **_expert_inputs(case, cfg, f, seed)}


def run(state: dict):
    if state["kind"] == "experts":
        e, epos = dec.experts(state["h"], state["ids"], state["wt"], state["wgu"], state["wd"])
        out = dec.SublayerOut(e=e, epos=epos, top=state["top"])
        hc = dec.Stream(state["inp"], state["mix"], state["out"])
        return {"h": dec.stream_step(state["x"], out, hc, state["inp"], state["norm"], state["cfg"].hidden, state["cfg"].rms_eps,
                                     torch.bfloat16, write_x=False)}
    eng = state["engine"]
    if state["kind"] == "scan":
        return _rows(eng.analyze(state["docs"]), state["index"])
    if state["kind"] == "prefill":
        reqs, logits = eng.given_start(state["prompts"], state["want"])
        for r in reversed(reqs):   # the next pass gets the same pages
            eng.given_end(r)
        return {"logits": logits, "keys": list(eng.kv.k), "values": list(eng.kv.v)}
    logits = eng.given_next(state["reqs"], state["next"])
    for r in state["reqs"]:   # the next pass tries the same token again
        r.output.pop()
    return {"logits": logits}


EVENTS = 50   # reported events of a log (``MatchEngine``'s default)


def _rows(results, index: dict) -> dict:
    """Analysis results as arrays: a log's reported events in their order, and their text."""
    out = _no_rows(len(results))
    for d, r in enumerate(results):
        for j, e in enumerate(r.events):
            out["line"][d, j], out["pattern"][d, j], out["score"][d, j] = e.line_number, index[e.matched_pattern.id], e.score
        out["total"][d], out["lines"][d] = r.summary.total_events, r.metadata["totalLines"]
        text = "\n".join(line for e in r.events for line in e.context).encode()[:out["context"].shape[1]]
        out["context"][d, :len(text)] = np.frombuffer(text, dtype=np.uint8)
    return out


def _no_rows(docs: int) -> dict:
    return {"line": np.full((docs, EVENTS), -1, dtype=np.int64), "pattern": np.full((docs, EVENTS), -1, dtype=np.int64),
            "score": np.zeros((docs, EVENTS)), "total": np.zeros(docs, dtype=np.int64), "lines": np.zeros(docs, dtype=np.int64),
            "context": np.zeros((docs, 4096), dtype=np.uint8)}


# ---------------------------------------------------------------- what a pass cannot do without
def _layer_work(cfg, i: int, tokens: int) -> tuple[int, int, int, int, int]:
    """Of layer i: (parameters a token uses, parameters ``tokens`` of them read, elements cached per
    token, multiply-adds per query and key at prefill, the same at decode)."""
    h = cfg.hidden
    if not hasattr(cfg, "layer_specs"):
        proj = h * (cfg.heads + 2 * cfg.kv_heads) * cfg.head_dim + cfg.heads * cfg.head_dim * h
        n = proj + 3 * h * cfg.intermediate
        return n, n, 2 * cfg.kv_heads * cfg.head_dim, 2 * cfg.heads * cfg.head_dim, 2 * cfg.heads * cfg.head_dim
    m, f = cfg.layer_specs[i].mixer, cfg.layer_specs[i].mlp
    use = 3 * h * (f.ff * max(1, f.top) + f.shared_ff) + h * f.experts
    read = 3 * h * (f.ff * (min(f.experts, tokens * f.top) if f.experts else 1) + f.shared_ff) + h * f.experts
    if isinstance(m, LatentSpec):
        own = h * (m.kv_rank + m.rot_dim) if m.kv_from < 0 else 0
        proj = h * (m.q_rank + m.heads) + own + m.q_rank * m.heads * (m.dim + m.rot_dim) + m.heads * m.vdim * h
        proj += m.heads * (m.dim + m.vdim) * m.kv_rank
        return (proj + use, proj + read, m.kv_rank + m.rot_dim, m.heads * (m.dim + m.rot_dim + m.vdim),
                m.heads * (2 * m.kv_rank + m.rot_dim))
    cached = m.kv_heads * (m.dim + m.vdim)
    proj = h * ((m.heads * m.dim + m.kv_heads * m.dim) + m.heads * m.vdim)
    proj += h * m.heads if m.conv else h * m.kv_heads * m.vdim   # values are the keys behind a convolution
    return proj + use, proj + read, cached, m.heads * (m.dim + m.vdim), m.heads * (m.dim + m.vdim)


def work(case: dict) -> dict:
    if case["kind"] == "scan":
        return {"bytes": float(case["docs"] * case["kib"] * 1024), "flops": 0.0}
    if case["kind"] == "experts":
        cfg, T = get_config(case["model"]), case["tokens"]
        f = cfg.layer_specs[1].mlp
        one = 3 * cfg.hidden * f.ff
        return {"bytes": float(2 * one * min(f.experts, T * f.top) + T * cfg.hidden * (2 + 4 * cfg.streams + 2) + 8 * T * f.top),
                "flops": float(2 * T * f.top * one)}
    cfg, lens, decode = _config(case), _lengths(case), case["kind"] == "decode"
    size = 4 if case["dtype"] == "float32" else 2
    tokens, rows = (len(lens) if decode else sum(lens)), len(lens)
    flops, byts = 2.0 * rows * cfg.hidden * cfg.vocab_size, 0.0
    byts += size * cfg.hidden * (cfg.vocab_size + tokens) + 4 * rows * cfg.vocab_size
    for i in range(cfg.layers):
        use, read, cached, pre, dec = _layer_work(cfg, i, tokens)
        w = getattr(cfg.layer_specs[i].mixer, "window", 0) if hasattr(cfg, "layer_specs") else 0
        if decode:
            seen = sum(min(n, w or n) for n in lens)
            keys = seen
        else:
            seen = sum((min(n, w or n) * (min(n, w or n) + 1)) // 2 + max(0, n - (w or n)) * w for n in lens)
            keys = tokens
        flops += 2.0 * tokens * use + 2.0 * seen * (dec if decode else pre)
        byts += read * (1 if case["weights"] == "fp8" else size) + size * cached * keys
    return {"bytes": float(byts), "flops": float(flops)}


def tolerance(case: dict):
    if case["kind"] == "scan":
        return {"rel": 2e-6}   # scores carry six digits; lines, patterns and text are whole
    if case.get("dtype") == "float32":
        return {"rel": 1e-5}   # 2.6e-6 from the 64-bit result
    if case["kind"] == "experts":
        return {"rel": 0.012}   # 0.3e-2 from it
    return {"rel": 0.03}   # bf16: 0.5e-2 to 0.8e-2 from it; fp8: rows whose rounding to e4m3 falls the other way


# ---------------------------------------------------------------- the same in 64 bits, plainly
def exact(case: dict, seed: int):
    if case["kind"] == "scan":
        return None if case["docs"] * case["kib"] > 4096 else _exact_scan(case, seed)
    if case["kind"] == "experts":
        return _exact_experts(case, seed)
    toks = [torch.tensor(t, device="cuda") for t in _tokens(case, seed)]
    with torch.no_grad():
        forward = {"sufolix": _exact_sufolix, "relurax": _exact_relurax}.get(get_config(case["model"]).arch, _exact_llama)
        return {"logits": torch.cat([forward(_config(case), _Weights(getattr(torch, case["dtype"])), toks[a:a + 24])
                                     for a in range(0, len(toks), 24)])}


def _exact_scan(case: dict, seed: int) -> dict:
    pats = synthetic_library(case["patterns"], seed=0).patterns
    find: dict = {}

    def matcher(m):
        src = re.escape(m.literal) if m.literal is not None else m.regex
        if src not in find:
            find[src] = re.compile(src, re.IGNORECASE if m.ignore_case else 0)
        return src

    prim = [matcher(p.primary) for p in pats]
    sec = [[matcher(s) for s in p.secondary] for p in pats]
    out = _no_rows(case["docs"])
    for d, doc in enumerate(_logs(case, seed)):
        starts = np.array([0] + [m.end() for m in re.finditer(b"\n", doc)])
        # a pattern never spans lines: what it finds in the whole log is what it finds line by line
        hits = {src: sorted({int(np.searchsorted(starts, m.start(), side="right")) - 1 for m in rx.finditer(doc)})
                for src, rx in find.items()}
        own = []
        for i, p in enumerate(pats):
            for line in hits[prim[i]]:
                bonus = 0.0
                for src, s in zip(sec[i], p.secondary):
                    near = min((abs(line - x) for x in hits[src]), default=None)
                    if near is not None and near <= s.window:
                        bonus += s.weight * (1 - near / (s.window + 1))
                score = p.primary.confidence * (1 + bonus) / (1 + sum(s.weight for s in p.secondary))
                own.append((-score, -p.severity_rank, line, i))
        own.sort()
        for j, (neg, _, line, i) in enumerate(own[:EVENTS]):
            out["line"][d, j], out["pattern"][d, j], out["score"][d, j] = line + 1, i, round(-neg, 6)
        out["total"][d], out["lines"][d] = len(own), len(starts)
    return {**out, "context": None}


class _Weights:
    """Random weights by name, as ``init_random`` draws them: a generator per name."""

    def __init__(self, dtype: torch.dtype):
        self.dtype = dtype

    def __call__(self, name: str, shape, std: float | None = None) -> torch.Tensor:
        g = torch.Generator(device="cuda")
        g.manual_seed(int.from_bytes(hashlib.sha256(f"{SAME_WEIGHTS}:{name}".encode()).digest()[:8], "little") & ((1 << 63) - 1))
        t = torch.randn(shape, generator=g, device="cuda", dtype=self.dtype)
        return t.mul_(std) if std is not None else t

    def scaled(self, name: str, shape) -> torch.Tensor:
        return (self(name, shape) * (1.0 / math.sqrt(shape[-1]))).double()


def _rms(x, eps, w=None):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if w is None else y * w


def _positions(toks) -> torch.Tensor:
    return torch.cat([torch.arange(t.numel(), device="cuda", dtype=torch.float64) for t in toks])


def _rotated(x, pos, base: float, dims: int, paired: bool):
    """Rotary positions on the first ``dims`` features of [T, H, D]: neighbours paired, or the halves."""
    inv = base ** (-torch.arange(0, dims, 2, device="cuda", dtype=torch.float64) / dims)
    c, s = (f(pos[:, None] * inv)[:, None] for f in (torch.cos, torch.sin))
    r = x[..., :dims]
    u, v = (r[..., 0::2], r[..., 1::2]) if paired else r.chunk(2, -1)
    y = (u * c - v * s, v * c + u * s)
    y = torch.stack(y, -1).flatten(-2) if paired else torch.cat(y, -1)
    return torch.cat([y, x[..., dims:]], -1)


def _attend(q, k, v, toks, scale: float, window: int = 0):
    """Causal attention of packed sequences, one kv head at a time."""
    out, a, per = [], 0, q.shape[1] // k.shape[1]
    for n in (t.numel() for t in toks):
        i = torch.arange(n, device="cuda")
        hidden = i[None, :] > i[:, None]
        if window:
            hidden |= i[:, None] - i[None, :] >= window
        o = torch.empty(n, q.shape[1], v.shape[2], device="cuda", dtype=torch.float64)
        for g in range(k.shape[1]):
            s = q[a:a + n, g * per:(g + 1) * per].transpose(0, 1) @ k[a:a + n, g].t().contiguous()
            p = torch.softmax((s * scale).masked_fill_(hidden, -math.inf), -1)
            o[:, g * per:(g + 1) * per] = (p @ v[a:a + n, g].contiguous()).transpose(0, 1)
        out.append(o)
        a += n
    return torch.cat(out)


def _head(x, toks, norm, eps, head):
    last = torch.tensor([t.numel() for t in toks], device="cuda").cumsum(0) - 1
    return _rms(x[last], eps, norm) @ head.double().t()


def _exact_llama(c, w: _Weights, toks):
    D, H, hid = c.head_dim, c.heads, c.hidden
    embed, pos = w("embed", (c.vocab_size, hid), 1.0), _positions(toks)
    x, T = embed[torch.cat(toks)].double(), sum(t.numel() for t in toks)
    std = 1.0 / math.sqrt(hid)

    def proj(h, i, n, rows, heads=None, s=std):
        y = h @ w(f"l{i}.w{n}", (rows, h.shape[1]), s).double().t()
        if heads is not None and c.qkv_bias:
            y = y + w(f"l{i}.b{n}", (rows,), 0.5).double()
        return y if heads is None else y.view(T, heads, D)

    for i in range(c.layers):
        h = _rms(x, c.rms_eps)
        q = _rotated(proj(h, i, "q", H * D, H), pos, c.rope_theta, D, False)
        k = _rotated(proj(h, i, "k", c.kv_heads * D, c.kv_heads), pos, c.rope_theta, D, False)
        o = _attend(q, k, proj(h, i, "v", c.kv_heads * D, c.kv_heads), toks, 1.0 / math.sqrt(D)).reshape(T, -1)
        x = x + proj(o, i, "o", hid, s=1.0 / math.sqrt(H * D))
        h = _rms(x, c.rms_eps)
        m = torch.nn.functional.silu(proj(h, i, "g", c.intermediate)) * proj(h, i, "u", c.intermediate)
        x = x + proj(m, i, "d", hid, s=1.0 / math.sqrt(c.intermediate))
    head = embed if c.tie_embeddings else w("lm_head", (c.vocab_size, hid), std)
    return _head(x, toks, None, c.rms_eps, head)


def _gated(h, w, p, ff: int, act):
    hid = h.shape[1]
    m = act(h @ w.scaled(p + "gate", (ff, hid)).t()) * (h @ w.scaled(p + "up", (ff, hid)).t())
    return m @ w.scaled(p + "down", (hid, ff)).t()


def _norm(w, name: str, n: int):
    return (1.0 + 0.1 * w(name, (n,))).double()


def _exact_experts(case: dict, seed: int) -> dict:
    cfg, f, raw = _expert_layer(case)
    i = _expert_inputs(case, cfg, f, seed)
    h, y = i["h"].double(), torch.zeros(case["tokens"], cfg.hidden, device="cuda", dtype=torch.float64)
    for e in range(f.experts):
        t, j = (i["ids"] == e).nonzero(as_tuple=True)
        u = h[t] * i["wt"][t, j][:, None].double()
        m = torch.nn.functional.silu(u @ raw["gate"][e].double().t()) * (u @ raw["up"][e].double().t())
        y.index_add_(0, t, m @ raw["down"][e].double().t())
    x = torch.einsum("tsw,sr->trw", i["x"].double(), i["mix"].double()) + i["out"].double()[None, :, None] * y[:, None]
    return {"h": _rms(torch.einsum("tsw,s->tw", x, i["inp"].double()), cfg.rms_eps, i["norm"].double())}


def _exact_sufolix(c, w: _Weights, toks):
    hid, S, T, pos = c.hidden, c.streams, sum(t.numel() for t in toks), _positions(toks)
    embed = w("embed", (c.vocab_size, hid))
    xs = (embed[torch.cat(toks)].double() * c.embed_scale)[:, None].repeat(1, S, 1)
    silu, first = torch.nn.functional.silu, None

    def streams(p):
        inp, out = (1.0 / S + 0.1 * w(p + "in", (S,))).double(), (1.0 + 0.1 * w(p + "out", (S,))).double()
        mix = w(p + "mix", (S, S))
        return inp, (0.05 * mix + torch.eye(S, dtype=mix.dtype, device="cuda")).double(), out

    for i, spec in enumerate(c.layer_specs):
        a, f, p = spec.mixer, spec.mlp, f"l{i}."
        inp, mix, out = streams(p + "hc1.")
        h = _rms(torch.einsum("tsw,s->tw", xs, inp), c.rms_eps, _norm(w, p + "norm1", hid))

        def heads(n, count, d):
            b = (0.2 * w(p + f"mix.{n}.b", (count * d,))).double()
            return (h @ w.scaled(p + "mix." + n, (count * d, hid)).t() + b).view(T, count, d)

        q, k = (_rms(_rotated(heads(n, cnt, a.dim), pos, a.rot_base, a.rot_dims, True), c.rms_eps)
                for n, cnt in (("q", a.heads), ("k", a.kv_heads)))
        v = heads("v", a.kv_heads, a.vdim)
        if a.v_mix and first is None:
            first = v
        elif a.v_mix:
            lam = (0.5 + 0.1 * w(p + "mix.vmix", (1,))).double()
            v = (1 - lam) * v + lam * first
        y = _attend(q, k, v, toks, a.scale).reshape(T, -1) @ w.scaled(p + "mix.o", (hid, a.heads * a.vdim)).t()
        xs = torch.einsum("tsw,sr->trw", xs, mix) + out[None, :, None] * y[:, None]
        inp, mix, out = streams(p + "hc2.")
        h = _rms(torch.einsum("tsw,s->tw", xs, inp), c.rms_eps, _norm(w, p + "norm2", hid))
        y = _gated(h, w, p + "mlp.", f.ff, silu)
        xs = torch.einsum("tsw,sr->trw", xs, mix) + out[None, :, None] * y[:, None]
    return _head(xs.sum(1), toks, _norm(w, "final.norm", hid), c.rms_eps, w.scaled("head", (c.vocab_size, hid)))


def _exact_relurax(c, w: _Weights, toks):
    hid, T, pos, eps = c.hidden, sum(t.numel() for t in toks), _positions(toks), c.rms_eps
    x, kept = w("embed", (c.vocab_size, hid))[torch.cat(toks)].double(), {}
    gelu = functools.partial(torch.nn.functional.gelu, approximate="tanh")

    def conv(u, taps):
        y, n = torch.zeros_like(u), taps.shape[1]
        for j in range(n):   # the tap ``back`` tokens before its own
            back = n - 1 - j
            prev = torch.zeros_like(u)
            prev[back:] = u[:T - back]
            prev[pos < back] = 0
            y += taps[:, j] * prev
        return y

    for i, spec in enumerate(c.layer_specs):
        a, f, p, q_ = spec.mixer, spec.mlp, f"l{i}.", f"l{i}.mix."
        h = _rms(x, eps, _norm(w, p + "norm1", hid))
        if isinstance(a, LatentSpec):
            src, R = (i if a.kv_from < 0 else a.kv_from), a.kv_rank
            if src == i:
                z = h @ w.scaled(q_ + "dkv", (R + a.rot_dim, hid)).t()
                kept[i] = (_rms(z[:, :R], eps, _norm(w, q_ + "dkv.norm", R)), _rotated(z[:, None, R:], pos, a.rot_base, a.rot_dim, False))
            lat, rot = kept[src]
            cq = _rms(h @ w.scaled(q_ + "dq", (a.q_rank, hid)).t(), eps, _norm(w, q_ + "dq.norm", a.q_rank))
            q = (cq @ w.scaled(q_ + "uq", (a.heads * (a.dim + a.rot_dim), a.q_rank)).t()).view(T, a.heads, -1)
            q = torch.cat([q[..., :a.dim], _rotated(q[..., a.dim:], pos, a.rot_base, a.rot_dim, False)], -1)
            k = torch.cat([(lat @ w.scaled(q_ + "uk", (a.heads * a.dim, R)).t()).view(T, a.heads, -1), rot.expand(T, a.heads, -1)], -1)
            o = _attend(q, k, (lat @ w.scaled(q_ + "uv", (a.heads * a.vdim, R)).t()).view(T, a.heads, -1), toks, a.scale)
        else:
            q, k = (conv(h @ w.scaled(q_ + n, (cnt * a.dim, hid)).t(), w.scaled(f"{q_}{n}.conv", (cnt * a.dim, a.conv))).view(T, cnt, a.dim)
                    for n, cnt in (("q", a.heads), ("k", a.kv_heads)))
            qn, kn = (_norm(w, f"{q_}{n}.norm", a.dim) for n in "qk")
            o = _attend(_rms(q, eps, qn), _rms(k, eps, kn), k, toks, a.scale, a.window)
        o = o * torch.sigmoid(h @ w.scaled(q_ + "g", (a.heads, hid)).t())[..., None]
        y = o.reshape(T, -1) @ w.scaled(q_ + "o", (hid, a.heads * a.vdim)).t()
        x = x + _rms(y, eps, _norm(w, p + "norm1b", hid))
        y = _gated(_rms(x, eps, _norm(w, p + "norm2", hid)), w, p + "mlp.", f.ff, gelu)
        x = x + _rms(y, eps, _norm(w, p + "norm2b", hid))
    return _head(x, toks, _norm(w, "final.norm", hid), eps, w.scaled("head", (c.vocab_size, hid)))
