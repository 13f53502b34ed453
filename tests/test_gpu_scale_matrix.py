"""Scaling of arrays long enough for the matrix-core form against the CPU path and against short calls:
numbers next to the edges of a step, exponents past the value, residues outside [0, m), ragged counts,
every array order, in place."""
import random

import numpy as np
import pytest

from grns_amd import largest_primes_below, product
from tests.helpers import to_res
from tests.test_gpu_scale_steps import _numbers

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _orders(x):
    n, count = x.shape
    wide = torch.zeros((n, count + 5), dtype=torch.int32, device="cuda")[:, 3:3 + count]
    rows = torch.zeros((count, n + 3), dtype=torch.int32, device="cuda")[:, 1:1 + n].t()
    spread = torch.zeros((n, 2 * count), dtype=torch.int32, device="cuda")[:, ::2]
    yield "moduli first", x.clone(), torch.empty_like(x)
    yield "numbers first", x.t().contiguous().t(), torch.empty((count, n), dtype=torch.int32, device="cuda").t()
    for name, view in (("odd row length", wide), ("padded rows", rows), ("every other column", spread)):
        view.copy_(x)
        yield name, view, view  # in place


@pytest.mark.parametrize("n", [1, 3, 8, 9, 16, 20, 32, 33, 50, 64])
def test_scale_long_arrays(n):
    import grns_amd as G
    from oracle.oracle import Oracle
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mod = largest_primes_below(n)
    count = 32768 + 8 * n + 13
    ctx, orc = G.Context(mod, 0), Oracle(mod)
    rnd = random.Random(n)
    M = product(mod)
    xs, Ds = _numbers(mod, 600, n) if n > 1 else ([], [])
    for bits in range(1, M.bit_length(), 7):
        xs.append(rnd.randrange(1 << (bits - 1), min(M, 1 << bits)))
        Ds.append(rnd.choice([0, 1, 30, rnd.randrange(2 * M.bit_length())]))
    xs += [0, 1, M - 1, M // 2]
    Ds += [5, 0, M.bit_length(), 31]
    for _ in range(200):
        xs.append(rnd.randrange(M))
        Ds.append(rnd.randrange(M.bit_length() + 100))
    base, D0 = to_res(xs, mod), np.array(Ds, np.uint32)
    off = np.array([17, 101, 333 % len(xs)])
    base[rnd.randrange(n), off] += np.array([0, mod[0] // 2, 0], np.int32)  # possibly past its modulus
    base[0, off[:1]] = -3
    D0[off] = 35
    pick = np.array([i % len(xs) for i in range(count)])
    x, D = np.ascontiguousarray(base[:, pick]), D0[pick]
    want = orc.scale2pow_array(base, D0)[:, pick]
    Dd = torch.from_numpy(D.view(np.int32)).cuda()
    xd = torch.from_numpy(x).cuda()
    short = torch.cat([ctx.scale2pow(xd[:, a:a + 16000].contiguous(), Dd[a:a + 16000])
                       for a in range(0, count, 16000)], dim=1).cpu().numpy()
    assert (short == want).all()
    for name, a, y in _orders(xd):
        ctx.scale2pow(a, Dd, y=y)
        assert (y.cpu().numpy() == want).all(), name
    orc.close()
    ctx.close()
