"""The sampler's workgroups per row: the token and its value do not depend on them."""
import pytest
import torch

from operator_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,vocab,ld", [(1, 4096, 4096), (1, 128256, 128256), (3, 5001, 5001), (7, 32000, 32064), (200, 9000, 9001)])
def test_parts_match_one_workgroup(dtype, rows, vocab, ld):
    torch.manual_seed(rows + vocab)
    x = torch.randn(rows, ld, device="cuda").to(dtype)[:, :vocab]
    x[0, vocab - 1] = x[0, 5] = x[0].max() + 1   # a tie: the smaller column wins
    temp = torch.rand(rows, device="cuda")
    temp[0] = 0
    if rows > 2:
        x[1] = float("-inf")
        x[2, ::3] = float("nan")
    seeds, pos = torch.arange(rows, device="cuda") + 5, torch.arange(rows, device="cuda") * 7
    assert ops.kernels().sample_parts(rows, vocab) > 1
    val, one_val = torch.empty(rows, device="cuda"), torch.empty(rows, device="cuda")
    tok = ops.sample(x, temp, seeds, pos, col_offset=11, out_val=val)
    one = torch.empty(rows, dtype=torch.long, device="cuda")
    ops.kernels().sample(x, temp, seeds, pos, one, 11, one_val)
    assert torch.equal(tok, one) and torch.equal(val, one_val) and int(tok[0]) == 16
