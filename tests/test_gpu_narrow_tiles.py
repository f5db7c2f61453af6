"""Both stages in one kernel with one or two columns a lane (4-byte types) or two (16-bit types): a few
columns of a wave and whole tiles, one wave per tile and up to eight, a last sub-row that is not whole, rows that
start at any element, odd numbers of buckets, rows that end by a list, by ties and through the
exact path of NaNs.  Bit-exact against the oracle: selection is a total order."""
import pytest
import torch

import oracle
from helpers import assert_same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.int32, torch.float16, torch.bfloat16, torch.int16],
                         ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("shape", [
    (1, 2048, 64, 2, 2),       # one row, 64 buckets, four waves or more per tile
    (3, 8192, 128, 4, 2),      # eight waves per tile
    (5, 5000, 320, 1, 2),      # a wave per tile, five tiles, the last sub-row not whole
    (129, 3002, 98, 1, 2),     # rows off 16 bytes, the last tile not whole
    (300, 7505, 142, 4, 4),    # three waves, or two, per tile; 142 buckets
    (1025, 2048, 64, 4, 2),    # more rows than the GPU holds at once
    (64, 20480, 512, 2, 2),    # eight tiles of one column a lane
    (4, 16384, 1024, 2, 2),    # eight tiles of two
])
def test_narrow_tiles(dtype, shape):
    from approx_topk import _native, topk
    from approx_topk.experimental import compact_indices
    rows, n, k, j, k_mult = shape
    g = torch.Generator().manual_seed(n + k + j)
    x = torch.randint(-30000, 30000, (rows, n), generator=g)
    if dtype.is_floating_point:
        x = x / 64
        x[0, ::3] = -0.0
        x[rows // 2, 7::997] = float("nan")
    x[rows - 1, n // 8:] = 5  # most candidates equal: the cut falls among them
    if rows > 2:
        x[1] = x[1].clamp(max=100)  # ties around the cut
    x = x.to(dtype)
    xd = x.cuda()
    plan = _native.describe(xd, k * k_mult, j, k)
    narrow = ("V=1,", "V=2,") if x.element_size() == 4 else ("V=2,",)
    assert plan.startswith("fused_regs_kernel") and any(v in plan for v in narrow), plan
    want = oracle.topk(x, k, -1, j=j, k_mult=k_mult)
    assert_same(*topk(xd, k, -1, j=j, k_mult=k_mult), *want, plan)
    only = compact_indices.topk_indices(xd, k, -1, j=j, k_mult=k_mult)
    assert torch.equal(only.cpu().long(), want[1]), plan



@pytest.mark.parametrize("dtype", [torch.float32, torch.float16], ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("shape", [
    (5, 5000, 320, 1, 2, 5008, 0),     # a wave per tile; rows on 16 bytes, some of them
    (129, 3002, 98, 1, 2, 3003, 1),    # rows anywhere
    (64, 20480, 512, 2, 2, 20484, 3),  # eight tiles of one column a lane
    (300, 7505, 142, 4, 4, 7600, 5),   # waves that share a tile
])
def test_narrow_tiles_of_rows_at_a_pitch(dtype, shape):
    from approx_topk import _native, topk
    rows, n, k, j, k_mult, pitch, first = shape
    g = torch.Generator().manual_seed(n + pitch)
    whole = (torch.randint(-30000, 30000, (rows, pitch), generator=g) / 64).to(dtype)
    whole[rows // 2, first + 7:first + n:997] = float("nan")
    whole[:, :first] = whole[:, first + n:] = float("inf")  # (between the rows: not theirs)
    x = whole[:, first:first + n]
    xd = whole.cuda()[:, first:first + n]
    plan = _native.describe(xd, k * k_mult, j, k)
    assert plan.startswith("fused_regs_kernel") and any(f"V={v}," in plan for v in (1, 2)), plan
    assert_same(*topk(xd, k, -1, j=j, k_mult=k_mult), *oracle.topk(x.contiguous(), k, -1, j=j, k_mult=k_mult), plan)
