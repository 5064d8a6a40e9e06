"""Given-token calls that come from different streams: what the engine keeps for a step (bucket state, the graph's logits,
cache pages) is not touched by the next call before the step has run."""
import contextlib

import pytest
import torch

from operator_amd.engine.llm import GenRequest, LLMEngine
from operator_amd.models.config import get_config
from operator_amd.models.kv_cache import PagedKVCache
from operator_amd.models.llama import LlamaModel

pytestmark = pytest.mark.gpu


def _calls(model, streams, late):
    """A step of three requests, another of three others (the same bucket), a new prompt on the pages of a request that
    ended, its step and a generated answer, each call on the next of ``streams``; ``late``: every call is queued behind a
    wait of some 10 ms."""
    kv = PagedKVCache.for_model(model, 16, 16)
    eng = LLMEngine(model, kv, max_batch=4, max_context=256, prefill_graphs=False, prefix_sharing=False)
    eng.warmup([4])
    n, out = 0, []

    @contextlib.contextmanager
    def call():
        nonlocal n
        with torch.cuda.stream(streams[n % len(streams)]):
            n += 1
            if late:
                torch.cuda._sleep(20_000_000)
            yield
        if not late:
            torch.cuda.synchronize()

    with call():
        reqs, lg = eng.given_start([list(range(3 + i, 20 + 5 * i)) for i in range(6)], [[0, 5]] * 6)
        out.append(lg)
    for t in range(3):
        for part in (reqs[:3], reqs[3:]):
            with call():
                out.append(eng.given_next(part, [100 + t, 7 * t, 900 - t]))
    eng.given_end(reqs[4])
    eng.given_end(reqs[5])
    with call():
        new, lg = eng.given_start([list(range(50, 110))], [[59]])
        out.append(lg)
    with call():
        out.append(eng.given_next([reqs[0], new[0]], [1, 2]))
    for r in (*reqs[:4], *new):
        eng.given_end(r)
    g = GenRequest(list(range(9, 60)), max_tokens=4, ignore_eos=True)
    with call():
        eng.generate([g])
    torch.cuda.synchronize()
    return [x.float().cpu() for x in out], g.output


@pytest.mark.parametrize("foreign", [False, True])
def test_calls_from_two_streams(foreign):
    m = LlamaModel(get_config("tiny-gqa4"), device="cuda").init_random(seed=5)
    torch.cuda.synchronize()
    want, tokens = _calls(m, [torch.cuda.default_stream()], False)
    own = [torch.cuda.Stream(), torch.cuda.Stream()]
    got, again = _calls(m, [own[0], torch.cuda.ExternalStream(own[1].cuda_stream) if foreign else own[1]], True)
    assert len(want) == len(got) == 9
    for a, b in zip(want, got):
        assert torch.equal(a, b)
    assert tokens == again
