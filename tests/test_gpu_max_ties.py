"""Arg-max among equal and nearly equal maxima spread over many blocks, in both array orders, against the
pipeline that compares mixed-radix digits."""
import random

import numpy as np
import pytest

from grns_amd import largest_primes_below, product
from tests.helpers import to_res

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n", [4, 8, 16, 32, 64])
@pytest.mark.parametrize("count", [3, 300, 70001, 400009])
def test_max_ties(n, count):
    import grns_amd as G
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mod = largest_primes_below(n)
    ctx, M, rnd = G.Context(mod, 0), product(mod), random.Random(n * count)
    rng = np.random.default_rng(count + n)
    for top in (M - 1, M // 2, M - (1 << 50), 3):
        near = [max(0, top - (d if top > 3 else d % 4)) for d in (0, 1, 2, 1000, 1 << 31, 1 << 45, 1 << 61, 0)]
        rows = to_res(near, mod)
        pick = rng.integers(0, len(near), count)
        x = rows[:, pick].astype(np.int32)
        low = rng.random(count) < 0.5  # the others: smaller values
        x[:, low] = to_res([rnd.randrange(max(1, top // 2)) for _ in range(16)], mod)[:, rng.integers(0, 16, int(low.sum()))]
        if low.all():
            x[:, 0] = rows[:, 0]
        xd = torch.from_numpy(x).cuda()
        want, at = ctx.max(xd, mrc=True)
        for a in (xd, xd.t().contiguous().t()):
            got, i = ctx.max(a)
            assert torch.equal(got, want) and int(i) == int(at), (top == M - 1, int(i), int(at))
            assert torch.equal(got, xd[:, int(i)])
    ctx.close()
