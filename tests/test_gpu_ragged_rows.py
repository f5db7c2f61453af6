"""Rows and sub-rows that start at any element: odd row lengths, odd pitches and bucket counts that
the load width does not divide, where the last lane of a row works on columns its neighbour has
too.  Bit-exact against the oracle (the reference's interleaved geometry,
priority_queue_approx_topk.cu:25-46): selection is a total order."""
import pytest
import torch

import oracle
from helpers import assert_same

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.float16, torch.bfloat16, torch.float64, torch.uint8, torch.int8]


def _data(rows, n, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    if dtype.is_floating_point:
        return (torch.randint(-300, 300, (rows, n), generator=g) / 16).to(dtype)  # ties in every bucket
    info = torch.iinfo(dtype)
    return torch.randint(info.min, info.max + 1, (rows, n), generator=g).to(dtype)


def _vec(dtype):
    return min(8, 16 // torch.empty(0, dtype=dtype).element_size())


@pytest.mark.parametrize("j", [1, 2, 3, 4])
@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d).split(".")[-1])
def test_bucket_counts_off_the_load_width(dtype, j):
    from approx_topk import _native, topk
    v = _vec(dtype)
    tile = 64 * v
    # one vector, a vector and one column, a tile less and more one column, three tiles less one; short
    # and long columns, a partial last sub-row of one element, of all but one, and none
    for b, length in ((v, 9), (v + 1, 300), (tile - 1, 37), (tile + 1, 6), (3 * tile - 1, 8)):
        for rem in (0, 1, b - 1):
            n = b * length + rem
            x = _data(3, n, dtype, 10 * b + j)
            want = oracle.topk(x, b * j, -1, j=j)
            assert_same(*topk(x.cuda(), b * j, -1, j=j), *want, f"b={b} n={n}")
            # the same rows in batches of 128 MiB, which keep the 16-byte loads unless their queues are long or
            # their buckets few
            xd = x.cuda().repeat((1 << 27) // (3 * n * x.element_size()) + 1, 1)
            if length in (37, 8) or j <= 2 and length in (300, 6):
                assert f"V={v}," in _native.describe(xd, b * j, j, b * j)
            values, indices = topk(xd, b * j, -1, j=j)
            assert_same(values[-3:], indices[-3:], *want, f"many rows, b={b} n={n}")


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d).split(".")[-1])
def test_padded_rows_off_the_load_width(dtype):
    from approx_topk.experimental import bucketed_argmax
    v = _vec(dtype)
    for n, k in ((64 * v * 5 + 3, 64 * v + 1), (1001, 77), (v * 3 + 1, v)):
        x = _data(5, n, dtype, n)
        got = bucketed_argmax.topk_triton(x.cuda(), k, -1, True)
        assert_same(*got, *oracle.bucketed_argmax(x, k, 1, interleaved=True), f"n={n} k={k}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16, torch.int8],
                         ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("shape", [
    (256, 10007, 64, 1, 8),     # both stages in one kernel, waves that share a tile
    (200, 12345, 1024, 2, 2),   # a wave per tile
    (130, 20001, 2048, 4, 2),   # several rounds of tiles or sixteen waves
    (3, 70001, 1000, 4, 2),     # few rows
    (2, 1 << 18 | 1, 50, 1, 2),  # slabs and the merge
])
def test_two_stages_of_odd_rows(dtype, shape):
    from approx_topk import topk
    rows, n, k, j, k_mult = shape
    x = _data(rows, n, dtype, n + j)
    want = oracle.topk(x, k, -1, j=j, k_mult=k_mult)
    assert_same(*topk(x.cuda(), k, -1, j=j, k_mult=k_mult), *want, str(shape))
    # the same rows in a matrix of even pitch, and in one that starts 4 bytes into a line
    es = x.element_size()
    wide = torch.zeros(rows, n + 17, dtype=dtype, device="cuda")
    wide[:, 4:4 + n] = x.cuda()
    assert_same(*topk(wide[:, 4:4 + n], k, -1, j=j, k_mult=k_mult), *want, f"view {shape} {4 * es}")


def test_nan_rows_off_the_load_width():
    from approx_topk import topk
    for dtype in (torch.float32, torch.bfloat16):
        for b, n, j in ((5 * 64 + 3, 20011, 2), (9, 5003, 4)):
            x = _data(4, n, dtype, b)
            x[1::2, ::97] = float("nan")
            x[0, 1::3] = -0.0
            assert_same(*topk(x.cuda(), b * j, -1, j=j), *oracle.topk(x, b * j, -1, j=j), f"b={b}")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.int16, torch.uint8, torch.int8],
                         ids=lambda d: str(d).split(".")[-1])
def test_views_that_start_off_four_bytes(dtype):
    """Two bytes into a line (16-bit elements), one and three (8-bit ones), with even and odd pitches: the kernels
    with loads of several elements take the address as they take the start of a row."""
    from approx_topk import _native, topk
    two_bytes = dtype.itemsize == 2
    v = 8
    cases = [  # rows, n, k, j, k_mult, interleaved, the kernel
        (256, 50003, 1001, 1, 1, True, f"J=1, V={v},"),                    # the last lane moves down
        (64, 1 << 17, 4096, 2, 1, True, f"J=2, V={v},"),
        (128, 70001, 4002, 2, 1, True, f"J=2, V={v},"),
        (2, 1 << 19, 50, 1, 2, True, "slabs"),
        (300, 4096, 256, 2, 2, True, "fused_"),                            # both stages in one kernel
        (300, 4099, 256, 1, 4, True, "fused_"),
        (7, 30011, 200, 2, 1, False, "split_bucket_kernel" if two_bytes else "contig_kernel"),
        (300, 8192, 256, 2, 4, False, "short contiguous" if two_bytes else "contig_kernel"),
    ]
    for rows, n, k, j, k_mult, interleaved, kernel in cases:
        x = _data(rows, n, dtype, n + j)
        if dtype.is_floating_point:
            x[0, ::97] = float("nan")
            x[1, ::3] = -0.0
        want = oracle.topk(x, k, -1, j=j, k_mult=k_mult, interleaved=interleaved)
        for pad, off in ((8, 1), (5, 1), (16, 3)):
            whole = torch.zeros(rows, n + pad, dtype=dtype, device="cuda")
            view = whole[:, off:off + n]
            view.copy_(x)
            assert view.data_ptr() % 4 != 0
            plan = _native.describe(view, k * k_mult, j, k, _native.INTERLEAVED if interleaved else _native.BALANCED)
            assert kernel in plan, plan
            assert_same(*topk(view, k, -1, j=j, k_mult=k_mult, interleaved=interleaved), *want, f"{plan} pad={pad} off={off}")
