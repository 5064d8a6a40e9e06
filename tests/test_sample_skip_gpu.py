"""Rows marked as not sampled get token 0 and leave the other rows' tokens as they are, on one workgroup a row and on several; a
plain NaN temperature stays greedy."""
import numpy as np
import pytest
import torch

from operator_amd import ops

DEV = "cuda"


@pytest.mark.gpu
@pytest.mark.parametrize("rows,vocab", [(1, 1000), (5, 32768), (240, 16384), (64, 128256)])
def test_skipped_rows(rows, vocab):
    assert ops.kernels().NO_SAMPLE_BITS == ops.NO_SAMPLE_BITS
    torch.manual_seed(rows)
    logits = torch.randn(rows, vocab, device=DEV).bfloat16()
    temp = np.linspace(0, 1.5, rows, dtype=np.float32)
    seeds, pos = torch.arange(rows, device=DEV), torch.arange(rows, device=DEV) * 7
    full = ops.sample(logits, torch.from_numpy(temp).to(DEV), seeds, pos)
    skip = np.arange(rows) % 3 == 0
    marked = temp.copy()
    marked.view(np.uint32)[skip] = ops.NO_SAMPLE_BITS
    logits[torch.from_numpy(skip).to(DEV)] = float("nan")
    val = torch.full((rows,), float("nan"), device=DEV)
    got = ops.sample(logits, torch.from_numpy(marked).to(DEV), seeds, pos, col_offset=64, out_val=val)
    want = ops.sample(logits, torch.from_numpy(temp).to(DEV), seeds, pos, col_offset=64)
    keep = torch.from_numpy(~skip).to(DEV)
    assert torch.equal(got[keep], want[keep]) and (got[~keep] == 64).all() and torch.isfinite(val).all()
    plain = ops.sample(logits, torch.from_numpy(marked).to(DEV), seeds, pos)
    assert torch.equal(plain[keep], full[keep]) and (plain[~keep] == 0).all()
    nan = torch.full((rows,), float("nan"), device=DEV)
    clean = torch.randn(rows, vocab, device=DEV).bfloat16()
    assert torch.equal(ops.sample(clean, nan, seeds, pos), ops.sample(clean, torch.zeros(rows, device=DEV), seeds, pos))
