"""scatter_rows_f32: a decode step's logits into the caller's rows."""
import pytest
import torch

from operator_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,n,cols,ld,off", [(1, 1, 5, 5, 0), (3, 7, 2048, 2048, 0), (5, 5, 2052, 2112, 0), (4, 9, 1000, 1003, 1), (2, 2, 4101, 4101, 0)])
def test_scatter_rows(dtype, rows, n, cols, ld, off):
    torch.manual_seed(cols)
    x = torch.randn(rows, ld, device="cuda").to(dtype)[:, off:off + cols] if ld >= off + cols else None
    out = torch.full((n, cols), 7.0, device="cuda")
    dst = torch.randperm(n)[:rows].int()
    dropped = rows > 1
    if dropped:
        dst[0] = -1
    ops.kernels().scatter_rows_f32(x, dst.cuda(), out)
    want = torch.full((n, cols), 7.0)
    for r, d in enumerate(dst.tolist()):
        if d >= 0:
            want[d] = x[r].float().cpu()
    assert torch.equal(out.cpu(), want)
