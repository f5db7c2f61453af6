"""Batches of few rows that take one-element loads where 16-byte loads are possible: aligned and odd
rows, with and without slabs, whole and padded, types of every width.  Bit-exact against the oracle:
selection is a total order."""
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


@pytest.mark.parametrize("dtype", [torch.uint8, torch.int8, torch.int64, torch.float64],
                         ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("shape", [
    (3, 38027, 560, 4, 1),       # one byte: seven eighths of the workgroups idle with 8-byte loads
    (2, 310384, 3196, 4, 1),     # slabs either way
    (14, 71905, 112, 2, 2),      # folded with wide loads, and the merge
])
def test_one_element_loads_of_one_and_eight_bytes(dtype, shape):
    from approx_topk import _native, topk
    rows, n, k, j, k_mult = shape
    g = torch.Generator().manual_seed(n + k)
    if dtype.is_floating_point:
        x = torch.randint(-3000, 3000, (rows, n), generator=g).to(dtype) / 16
        x[0, ::3] = -0.0
        x[1, ::9973] = float("nan")
    else:
        info = torch.iinfo(dtype)
        x = torch.randint(max(info.min, -3000), min(info.max, 3000) + 1, (rows, n), generator=g).to(dtype)
        x[1, ::97] = info.min
    xd = x.cuda()
    plan = _native.describe(xd, k * k_mult, j, k)
    assert "V=1," in plan, plan
    assert_same(*topk(xd, k, -1, j=j, k_mult=k_mult), *oracle.topk(x, k, -1, j=j, k_mult=k_mult), plan)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.int8, torch.float64],
                         ids=lambda d: str(d).split(".")[-1])
def test_one_element_loads_of_padded_rows(dtype):
    from approx_topk import _native
    from approx_topk.experimental import bucketed_argmax
    g = torch.Generator().manual_seed(11)
    for rows, n, k in ((3, 50001, 1000), (2, 70003, 640), (1, 1001, 333)):
        x = torch.randint(-120, 120, (rows, n), generator=g).to(dtype)
        plan = _native.describe(x.cuda(), k, 1, k, _native.INTERLEAVED_PADDED)
        assert "V=1," in plan, plan
        got = bucketed_argmax.topk_triton(x.cuda(), k, -1, True)
        assert_same(*got, *oracle.bucketed_argmax(x, k, 1, interleaved=True), f"n={n} k={k}")
