"""Short evaluations, comparisons and divisions (a wave group per number) against long ones (a lane per
number, rare numbers behind): uniform numbers, numbers near 0 and M, residues outside [0, m), with the
rare queue's options."""
import random

import numpy as np
import pytest

from grns_amd import largest_primes_below, product
from tests.helpers import to_res

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _numbers(mod, count, seed):
    rng = np.random.default_rng(seed)
    n, M = len(mod), product(mod)
    x = np.stack([rng.integers(0, m, count) for m in mod]).astype(np.int32)
    near = [0, 1, 2, M - 1, M - 2, M // 2, M // 2 + 1]
    near += [(1 << k) - 1 for k in range(2, M.bit_length() - 1, 5)]
    near += [M - (1 << k) for k in range(2, M.bit_length() - 1, 5)]
    edges = to_res(near, mod)
    at = np.unique(rng.integers(0, count, 40 + count // 50))
    x[:, at] = edges[:, at % edges.shape[1]]
    off = np.unique(rng.integers(0, count, 20 + count // 300))
    x[rng.integers(0, n, off.size), off] -= mod[0]  # outside [0, m)
    return torch.from_numpy(x).cuda()


@pytest.mark.parametrize("n", [1, 2, 3, 4, 8, 11, 16, 27, 32, 45, 64])
def test_short_and_long_calls(n):
    import grns_amd as G
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mod = largest_primes_below(n)
    ctx = G.Context(mod, 0)
    group = 1 << (n - 1).bit_length()
    lanes = 4096 * torch.cuda.get_device_properties(0).multi_processor_count
    count = lanes // group + 77
    x, y = _numbers(mod, count, n), _numbers(mod, count, n + 100)
    y[:, ::3] = x[:, ::3]
    ops = [lambda a, b: ctx.eval(a), lambda a, b: ctx.eval(a, fast=True), lambda a, b: ctx.cmp(a, b)]
    for staging, spread in ((True, True), (False, True), (True, False)):
        ctx.rare_staging(staging)
        ctx.rare_spread(spread)
        for k, op in enumerate(ops):
            want = op(x, y).contiguous().view(torch.int32)
            step = lanes // group // 3 + 1
            got = torch.cat([op(x[:, a:a + step], y[:, a:a + step]) for a in range(0, count, step)])
            assert torch.equal(got.contiguous().view(torch.int32), want), (k, staging, spread)
            assert torch.equal(op(x[:, 5:6], y[:, 5:6]).contiguous().view(torch.int32).flatten(),
                               want.view(count, -1)[5]), k
    ctx.close()


@pytest.mark.parametrize("n", [2, 4, 8, 20, 32, 64])
def test_short_divisions(n):
    """Quotients and remainders of pairs of every length."""
    import grns_amd as G
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mod = largest_primes_below(n)
    ctx = G.Context(mod, 0)
    top = product(mod).bit_length() - 3
    rnd = random.Random(n)
    xs = [rnd.randrange(1 << rnd.randrange(1, top)) for _ in range(203)]
    ds = [max(1, x >> rnd.randrange(40)) for x in xs]
    x, d = to_res(xs, mod), to_res(ds, mod)
    x, d = torch.from_numpy(x).cuda(), torch.from_numpy(d).cuda()
    want_q = to_res([a // b for a, b in zip(xs, ds)], mod)
    want_r = to_res([a % b for a, b in zip(xs, ds)], mod)
    m = np.array(mod, np.int32)[:, None]
    for fast in (False, True):
        q, r = ctx.div(x, d, fast=fast)
        q, r = q.cpu().numpy(), r.cpu().numpy()
        assert (r == want_r).all(), fast
        assert ((q == want_q) | ((q == m) & (want_q == 0))).all(), fast
    ctx.close()
