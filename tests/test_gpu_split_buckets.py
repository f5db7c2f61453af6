"""Contiguous buckets that adjacent lanes share, a piece of at most 64 bytes each and turn by turn when
there are more pieces than lanes.  Bit-exact against the oracle (the reference's contiguous bucket
geometry, priority_queue_approx_topk.cu:47-54): selection is a total order."""
import pytest
import torch

import oracle
from helpers import assert_same

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.int32, torch.float16, torch.bfloat16, torch.int16]


def _data(rows, n, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    if dtype.is_floating_point:
        x = (torch.randint(-300, 300, (rows, n), generator=g) / 16).to(dtype)  # ties in every bucket
        x[0, ::3] = -0.0
        x[1, n // 5:] = float("-inf")        # buckets of nothing else
        x[-1, ::97] = float("nan")           # and a row that goes through the order keys
        return x
    info = torch.iinfo(dtype)
    x = torch.randint(info.min, info.max + 1, (rows, n), generator=g).to(dtype)
    x[1, n // 5:] = info.min
    return x


def _check(x, k, j, k_mult=1, view=False):
    from approx_topk import _native, topk
    rows, n = x.shape
    xd = x.cuda()
    if view:  # rows that start 4 bytes into a line, spaced by an odd pitch
        wide = torch.zeros(rows, n + 7, dtype=x.dtype, device="cuda")
        at = 4 // x.element_size()
        wide[:, at:at + n] = xd
        xd = wide[:, at:at + n]
    plan = _native.describe(xd, k * k_mult, j, k, _native.BALANCED)
    assert plan.startswith("split_bucket_kernel<"), plan
    assert_same(*topk(xd, k, -1, j=j, k_mult=k_mult, interleaved=False),
                *oracle.topk(x, k, -1, j=j, k_mult=k_mult, interleaved=False), f"{plan} {x.dtype} n={n}")


@pytest.mark.parametrize("j", [1, 2, 3, 4])
@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d).split(".")[-1])
def test_buckets_shared_by_lanes(dtype, j):
    per = 64 // torch.empty(0, dtype=dtype).element_size()  # elements of a piece
    # bucket lengths around one, two and 64 pieces, and past two turns; some buckets one longer, all
    # but one longer, and none
    for m in (per, per + 1, 2 * per - 1, 2 * per, 2 * per + 1, 5 * per + 3, 64 * per - 1, 64 * per, 64 * per + 1, 150 * per):
        b = 5 if m > 8 * per else 37
        for r in (0, 1, b - 1):
            if r == 0 and m % 2 == 0:
                m += 1  # (buckets of whole packs take another kernel)
            _check(_data(4, b * m + r, dtype, m + j), b * j, j, view=r == 1)


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d).split(".")[-1])
def test_buckets_shorter_than_a_piece(dtype):
    least = 16 // torch.empty(0, dtype=dtype).element_size()  # one load
    for m, j in ((least, 1), (least, 2), (least + 1, 2), (4 * least - 1, 2), (16, 4)):
        b = 16384 // 4 + 3
        _check(_data(4, b * m + 11, dtype, m), b * j, j, view=m == least + 1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16], ids=lambda d: str(d).split(".")[-1])
def test_split_buckets_with_a_second_stage_and_narrow_results(dtype):
    from approx_topk.experimental import compact_indices
    x = _data(5, 30011, dtype, 7)
    _check(x, 100, 2, k_mult=4)
    want = oracle.topk(x, 200, -1, j=2, interleaved=False)
    v, i = compact_indices.topk(x.cuda(), 200, -1, j=2, interleaved=False)
    assert i.dtype == torch.int32
    assert_same(v, i.long(), *want)
    only = compact_indices.topk_indices(x.cuda(), 200, -1, j=2, interleaved=False)
    assert torch.equal(only.cpu().long(), want[1])


def test_longest_split_bucket_and_few_of_them():
    from approx_topk import _native
    for m, b, split in ((16383, 256, True), (16384, 256, False), (16383, 255, False), (8190, 1, True), (8192, 1, False)):
        text = _native.describe(torch.empty(2, m * b + 1, device="cuda"), b, 1, b, _native.BALANCED)
        assert text.startswith("split_bucket_kernel") == split, (m, b, text)
    _check(_data(2, 16383 * 256 + 1, torch.float32, 3), 512, 2)
