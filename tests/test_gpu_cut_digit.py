"""The select of the one-kernel path where its cut digit (the leading eleven bits of a key) holds a planned number of
candidates, of which a planned number is wanted: none left out, the list's 64 and one around it, more than it
takes.  A wave per tile and two to eight that share one, so that the first digits are counted after a scan and after
a fold, with loads of every width.  Bit-exact against the oracle: selection is a total order."""
import pytest
import torch

import oracle
from helpers import assert_same

pytestmark = pytest.mark.gpu

ROWS = sorted({(count, need) for count in (1, 2, 63, 64, 65, 66, 130) for need in (1, (count + 1) // 2, max(1, count - 1), count)})

# (the rest of a bucket, candidates below the digit, in it, above it): ranges of each type, [from, below)
RANGES = {
    torch.float32: ((-900, -100), (-50, 0.25), (1, 1.25), (2, 900)),
    torch.float64: ((-900, -100), (-50, 0.25), (1, 1.25), (2, 900)),
    torch.float16: ((-900, -100), (-50, 0.25), (1, 1.03125), (2, 900)),
    torch.int32: ((-1 << 30, -1 << 24), (-1 << 20, 0), (0, 1 << 21), (1 << 21, 1 << 30)),
    torch.int16: ((-30000, -20000), (-10000, 0), (0, 32), (32, 30000)),
}


def _uniform(shape, bounds, dtype, g):
    low, high = bounds
    if not dtype.is_floating_point:
        return torch.randint(low, high, shape, generator=g).to(dtype)
    x = (low + (high - low) * torch.rand(shape, generator=g, dtype=torch.float64)).to(dtype)
    return torch.where(x >= high, torch.full_like(x, low), x)  # (rounded up to the bound)


# (n, k0, j, columns a lane, waves per tile)
SHAPES = {
    torch.float32: [(8192, 512, 1, 1, 1), (8192, 512, 2, 1, 2), (32768, 512, 2, 2, 4), (65536, 512, 1, 4, 4), (65536, 512, 4, 2, 8)],
    torch.int32: [(8192, 512, 4, 1, 4), (16384, 512, 1, 2, 2), (8192, 2048, 1, 4, 1)],
    torch.float16: [(8192, 512, 1, 2, 2), (8192, 512, 4, 2, 8), (8192, 2048, 1, 4, 1), (65536, 512, 1, 4, 4)],
    torch.int16: [(8192, 512, 2, 2, 4), (65536, 1024, 1, 4, 2)],
    torch.float64: [(8192, 512, 1, 2, 2), (8192, 512, 4, 2, 8), (8192, 1024, 1, 2, 1)],
}


@pytest.mark.parametrize("dtype", SHAPES, ids=lambda d: str(d)[6:])
def test_cut_digit(dtype):
    from approx_topk import _native, topk
    rest, below, inside, above = RANGES[dtype]
    for n, k0, j, vec, split in SHAPES[dtype]:
        k, b = k0 // 2, k0 // j
        g = torch.Generator().manual_seed(n + k0 + j)
        x = _uniform((len(ROWS), n // b, b), rest, dtype, g)
        for row, (count, need) in enumerate(ROWS):
            best = torch.cat([_uniform((k - need,), above, dtype, g), _uniform((count,), inside, dtype, g),
                              _uniform((k0 - (k - need) - count,), below, dtype, g)])
            places = torch.rand(b, n // b, generator=g).argsort(1)[:, :j]  # j sub-rows of every bucket
            x[row, places.T.reshape(-1), torch.arange(b).repeat(j)] = best[torch.randperm(k0, generator=g)]
        x = x.reshape(len(ROWS), n)
        xd = x.cuda()
        plan = _native.describe(xd, k0, j, k)
        assert plan.startswith("fused_regs_kernel") and f"V={vec}," in plan and f"split={split} " in plan, plan
        assert_same(*topk(xd, k, -1, j=j, k_mult=2), *oracle.topk(x, k, -1, j=j, k_mult=2), plan)
