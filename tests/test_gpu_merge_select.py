"""Rows cut into slabs whose merge takes the second stage along.  Bit-exact against the oracle (the
reference's interleaved geometry and its second stage, priority_queue.py:85-88): selection is a total order."""
import pytest
import torch

import oracle
from helpers import assert_same

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.float16, torch.bfloat16, torch.int32, torch.int16, torch.uint8]


def _data(rows, n, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    if dtype.is_floating_point:
        x = (torch.randint(-4000, 4000, (rows, n), generator=g) / 16).to(dtype)
        x[0] = x[0].clamp(min=0) * (x[0] > 240).to(dtype)   # zeros of both signs at the cut
        x[0, ::5] = -0.0
        x[-1, ::9973] = float("nan")
        x[-1, 1::3] = float("-inf")
        return x
    info = torch.iinfo(dtype)
    return torch.randint(info.min, info.max + 1, (rows, n), generator=g).to(dtype)


# (rows, n, k, j, k_mult): one bucket; a handful; 256 candidates and 257 and more (ranked by counting, by radix
# passes); as many buckets as threads and more; the most candidates and one bucket more than that
SHAPES = [
    (2, 1 << 20, 2, 4, 2, True), (3, 600011, 10, 2, 4, True), (2, 1 << 20, 128, 1, 2, True),
    (2, 1 << 20, 129, 2, 2, True), (2, (1 << 20) + 77, 100, 3, 3, True), (1, 200003, 300, 4, 4, True),
    (2, 1 << 20, 1024, 1, 2, True), (1, 1 << 20, 512, 1, 4, True), (1, 1 << 20, 1025, 1, 2, False),
]


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d).split(".")[-1])
def test_merge_with_the_second_stage(dtype):
    from approx_topk import _native, topk
    from approx_topk.experimental import compact_indices
    for rows, n, k, j, k_mult, taken in SHAPES:
        x = _data(rows, n, dtype, n + k)
        xd = x.cuda()
        plan = _native.describe(xd, k * k_mult, j, k)
        assert ("stream_merge_select_kernel" in plan) == taken, plan
        want = oracle.topk(x, k, -1, j=j, k_mult=k_mult)
        assert_same(*topk(xd, k, -1, j=j, k_mult=k_mult), *want, plan)
        only = compact_indices.topk_indices(xd, k, -1, j=j, k_mult=k_mult)
        assert only.dtype == torch.int32 and torch.equal(only.cpu().long(), want[1]), plan


def test_merge_with_the_second_stage_of_equal_rows():
    from approx_topk import topk
    for k, j, k_mult in ((100, 2, 2), (500, 4, 4)):   # nothing but the indices decides
        x = torch.zeros(2, 1 << 20)
        x[1] = float("nan")
        assert_same(*topk(x.cuda(), k, -1, j=j, k_mult=k_mult), *oracle.topk(x, k, -1, j=j, k_mult=k_mult), f"{k}")
