"""Rows cut into fewer slabs than there were waves to ask for (no more workgroups than CUs) or into more (a workgroup a
CU), and their merges of four partial queues a thread in many workgroups: slabs of uneven lengths, down to two of them
and up to 145, folded columns, both widths of loads, with the second stage in the merge and behind it, rows that start
anywhere.  Bit-exact against the oracle: selection is a total order."""
import re

import pytest
import torch

import oracle
from helpers import assert_same

pytestmark = pytest.mark.gpu

F64, F32, F16, BF16, I32, I8 = (torch.float64, torch.float32, torch.float16, torch.bfloat16, torch.int32, torch.int8)

# (type, rows, n, k, j, k_mult, slabs asked for by the waves alone, slabs taken)
CUT = [
    (BF16, 5, 241799, 144, 2, 1, 26, 25), (I8, 2, 1568123, 384, 1, 1, 22, 21), (F64, 3, 1250960, 72, 2, 1, 86, 85),
    (F64, 44, 124526, 132, 2, 1, 6, 5), (I32, 9, 552192, 336, 4, 1, 29, 28), (BF16, 3, 423452, 36, 2, 4, 43, 42),
    (F32, 48, 117143, 72, 1, 4, 3, 2), (I32, 33, 154094, 264, 4, 4, 4, 3),
]
RAISED = [
    (F64, 1, 577600, 132, 4, 2, 64, 68), (F64, 15, 129856, 744, 3, 1, 3, 4), (F32, 3, 1205184, 2220, 3, 1, 4, 6),
    (F64, 1, 1121152, 96, 4, 1, 72, 145), (F64, 24, 163615, 36, 3, 2, 6, 10), (BF16, 64, 143862, 24, 2, 2, 2, 4), (F16, 41, 285696, 36, 2, 2, 4, 6),
    (I32, 6, 550208, 144, 4, 1, 34, 42), (F32, 70, 61376, 24, 4, 2, 2, 3), (F32, 11, 209437, 408, 1, 2, 2, 4),
    (F16, 27, 188992, 168, 1, 4, 2, 4), (I32, 2, 6448512, 72, 4, 2, 89, 128), (I32, 25, 417312, 744, 4, 2, 4, 5),
]


@pytest.mark.parametrize("call", CUT + RAISED, ids=lambda c: f"{str(c[0])[6:]}-{c[1]}x{c[2]}-{c[6]}to{c[7]}")
def test_slabs(call):
    from approx_topk import _native, topk
    from approx_topk.experimental import compact_indices
    dtype, rows, n, k, j, k_mult, _, slabs = call
    g = torch.Generator().manual_seed(n + k + j)
    x = torch.randint(-127, 128, (rows, n), generator=g) if dtype == I8 else torch.randint(-30000, 30000, (rows, n), generator=g)
    if dtype.is_floating_point:
        x = x / 64
        x[0, ::3] = -0.0
        if rows > 2:
            x[rows // 2, 7::9973] = float("nan")
    x[rows - 1, n // 8:] = 5  # equal elements in every slab but the first: the lower index wins
    x = x.to(dtype)
    xd = x.cuda()
    plan = _native.describe(xd, k * k_mult, j, k)
    assert "stream_merge" in plan and re.search(r"slabs=(\d+)", plan)[1] == str(slabs), plan
    want = oracle.topk(x, k, -1, j=j, k_mult=k_mult)
    assert_same(*topk(xd, k, -1, j=j, k_mult=k_mult), *want, plan)
    only = compact_indices.topk_indices(xd, k, -1, j=j, k_mult=k_mult)
    assert torch.equal(only.cpu().long(), want[1]), plan
