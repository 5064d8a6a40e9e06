"""The sampler's workgroups per row: the token and its value do not depend on them."""
import pytest
import torch

from operator_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,vocab,ld", [(1, 16384, 16384), (1, 128256, 128256), (3, 16401, 16401), (7, 32000, 32064), (200, 98400, 98401)])
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


@pytest.mark.parametrize("rows,vocab,parts", [(1, 16383, 1), (1, 16384, 8), (64, 16384, 8), (65, 28671, 1), (65, 28672, 14), (160, 28672, 12),
                                              (161, 98303, 1), (161, 98304, 12), (224, 98304, 9), (225, 152064, 1), (8, 4096, 1)])
def test_rows_and_columns_that_take_parts(rows, vocab, parts):
    """Where several workgroups and the merge were measured faster than one."""
    assert ops.kernels().sample_parts(rows, vocab) == parts
