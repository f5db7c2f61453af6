"""Batches of few rows that take one-element loads where 16-byte loads are possible: aligned and odd
rows, with and without slabs, whole and padded.  Bit-exact against the oracle: selection is a total order."""
import pytest
import torch

import oracle
from helpers import assert_same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.int32, torch.float16, torch.bfloat16, torch.int16],
                         ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("shape", [
    (2, 1 << 18, 4096, 4, 2),    # CUs left idle, no merge
    (3, 100003, 1560, 2, 1),     # small batches, odd rows
    (2, 1 << 20, 2048, 4, 1),    # slabs either way
    (5, 1 << 20, 512, 2, 2),     # folded with 16-byte loads
])
def test_one_element_loads(dtype, shape):
    from approx_topk import _native, topk
    rows, n, k, j, k_mult = shape
    g = torch.Generator().manual_seed(n + k)
    x = torch.randint(-3000, 3000, (rows, n), generator=g)
    if dtype.is_floating_point:
        x = x / 16
        x[0, ::3] = -0.0
        x[1, ::9973] = float("nan")
    x = x.to(dtype)
    xd = x.cuda()
    plan = _native.describe(xd, k * k_mult, j, k)
    assert "V=1," in plan, plan
    assert_same(*topk(xd, k, -1, j=j, k_mult=k_mult), *oracle.topk(x, k, -1, j=j, k_mult=k_mult), plan)
