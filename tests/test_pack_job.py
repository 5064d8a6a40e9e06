"""PackJob: documents in the scan's layout, copied in pieces by several threads (past the caches from 8 MB on) while the caller
already uploads the first of them."""
import numpy as np
import pytest

from operator_amd.ops import patterns

PIECE = 256 << 10


def _packed(docs, seg):
    return b"".join(d + b"\0" * (-(len(d) + 1) % seg + 1) for d in docs)


# empty documents, edges of segments and pieces; below and past 8 MB (copies past the caches); a destination off 16 bytes
@pytest.mark.parametrize("big", [0, 9 << 20])
@pytest.mark.parametrize("seg,threads,shift", [(64, 1, 0), (64, 5, 0), (1024, 16, 0), (256, 3, 8), (64, 2, 1)])
def test_pieces_make_the_layout(big, seg, threads, shift):
    P, rng = patterns(), np.random.default_rng(seg + threads + big)
    sizes = [0, 1, seg - 1, seg, seg + 1, PIECE - 1, PIECE, PIECE + 1, 0, 2 * PIECE + 77, big, 5]
    docs = [rng.integers(0, 256, n, dtype=np.uint8).tobytes() for n in sizes]
    total, first = P.plan_docs(sizes, seg)
    want = _packed(docs, seg)
    assert len(want) == total
    buf = np.full(total + 64, 0xEE, dtype=np.uint8)
    at = (-buf.ctypes.data) % 16 + shift
    job = P.PackJob(docs, first, seg, buf.ctypes.data + at, threads)
    for n in (0, 1, 6, len(docs)):   # in place as far as waited for
        job.wait(n)
        assert buf[at:at + first[n] * seg].tobytes() == want[:first[n] * seg]
    job.close()
    assert (buf[at + total:] == 0xEE).all() and (buf[:at] == 0xEE).all()


def test_a_closed_job_copies_no_further():
    P, docs = patterns(), [b"x" * (1 << 20)] * 16
    total, first = P.plan_docs([len(d) for d in docs], 64)
    buf = np.zeros(total, dtype=np.uint8)
    job = P.PackJob(docs, first, 64, buf.ctypes.data, 1)
    job.wait(2)
    job.close()
    with pytest.raises(RuntimeError):
        job.wait(16)
    assert not buf[first[3] * 64:].any()
    with pytest.raises(IndexError):
        job.wait(17)
    with pytest.raises(ValueError):
        P.PackJob(docs, first[:-1], 64, buf.ctypes.data, 1)
    with pytest.raises(ValueError):   # a plan for shorter documents
        P.PackJob(docs, [i for i in range(17)], 64, buf.ctypes.data, 1)
