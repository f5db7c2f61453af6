"""Columns of 33-64 sub-rows of 16-bit elements in launches of thousands of workgroups, whose waves
have all loads of a short run under way at once: every length of the odd batch before the whole
ones.  Bit-exact against the oracle on sample rows (a row's result depends on that row alone)."""
import pytest
import torch

import oracle
from helpers import assert_same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("j", [2, 4])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.int16], ids=lambda d: str(d).split(".")[-1])
def test_short_columns(dtype, j):
    from approx_topk import _native, topk
    rows, b = 2048, 512
    sample = torch.tensor([0, 1, 1023, rows - 1])
    for full in (33, 34, 37, 40, 43, 46, 49, 52, 55, 58, 61, 63):
        n = full * b + (full % 3) * 100
        g = torch.Generator(device="cuda").manual_seed(full)
        x = torch.randint(-300, 300, (rows, n), generator=g, device="cuda").to(dtype)   # ties in every column
        if dtype.is_floating_point:
            x[1, ::301] = float("nan")
            x[rows - 1] = x[rows - 1].clamp(max=0) * 0.0                                # zeros of both signs
        plan = _native.describe(x, b * j, j, b * j)
        assert "U=8" in plan and "RUN=0" in plan and plan.endswith("wave-stores"), plan
        v, i = topk(x, b * j, -1, j=j)
        assert_same(v[sample.cuda()], i[sample.cuda()], *oracle.topk(x[sample.cuda()].cpu(), b * j, -1, j=j), plan)
