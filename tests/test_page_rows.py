"""Page lists of a decode batch into the bytes of its table: what numpy's assignment row by row gives, and what is refused."""
import numpy as np
import pytest
import torch

from operator_amd import ops


@pytest.mark.parametrize("rows,cols,head", [(1, 1, 0), (3, 5, 8), (64, 512, 3076)])
def test_page_rows(rows, cols, head):
    rng = np.random.default_rng(rows)
    lists = [rng.integers(-1, 2 ** 31, rng.integers(0, cols + 1)).tolist() for _ in range(rows)]
    lists[0] = list(range(cols))   # a full row
    lists[-1] = [np.int64(v) for v in lists[-1]]
    buf = torch.full((head + 4 * (rows + 1) * cols,), 7, dtype=torch.uint8)
    want = buf[head:].clone().numpy().view(np.int32).reshape(rows + 1, cols)
    for i, pages in enumerate(lists):
        want[i, :len(pages)] = pages
    ops.kernels().page_rows(buf, head, cols, lists)
    assert (buf[head:].numpy().view(np.int32).reshape(rows + 1, cols) == want).all() and (buf[:head] == 7).all()


def test_page_rows_refuses():
    C, t = ops.kernels(), torch.zeros(64, dtype=torch.uint8)
    C.page_rows(t, 0, 4, [])
    C.page_rows(t, 64, 4, [])
    for table, lists, err in ((t, [[0] * 5], RuntimeError), (t, [[1]] * 5, RuntimeError), (t, [[2 ** 31]], RuntimeError), (t, [(1, 2)], RuntimeError),
                              (t, [["a"]], TypeError), (t[1:], [[1]], RuntimeError), (t[::2], [[1]], RuntimeError), (t.int(), [[1]], RuntimeError)):
        with pytest.raises(err):
            C.page_rows(table, 0, 4, lists)
    for at, cols in ((4, 16), (-4, 4), (2, 4), (68, 4), (0, 0)):
        with pytest.raises(RuntimeError):
            C.page_rows(t, at, cols, [[1]])


def test_slots_of_the_positions():
    rows, cols, P = 5, 6, 16
    buf = torch.zeros(8 + 2 * rows * 8 + rows * cols * 4, dtype=torch.uint8)
    n = buf.numpy()
    pos, slots = n[8:8 + 8 * rows].view(np.int64), n[8 + 8 * rows:8 + 16 * rows].view(np.int64)
    pos[:] = [0, 15, 16, 95, 200]   # the last one past the table: its last page
    lists = [[3], [4], [5, 6], list(range(10, 16)), list(range(20, 26))]
    ops.kernels().page_rows(buf, 8 + 16 * rows, cols, lists, P, 8, 8 + 8 * rows)
    assert slots.tolist() == [48, 79, 96, 15 * 16 + 15, 25 * 16 + 8]
    for page_size, at, to in ((-1, 8, 48), (16, -8, 48), (16, 4, 48), (16, 8, 180), (16, 8, 49)):
        with pytest.raises(RuntimeError):
            ops.kernels().page_rows(buf, 8 + 16 * rows, cols, lists, page_size, at, to)
    pos[1] = -1
    with pytest.raises(RuntimeError):
        ops.kernels().page_rows(buf, 8 + 16 * rows, cols, lists, P, 8, 48)
