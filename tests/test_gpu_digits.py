"""Mixed-radix digits of the per-lane conversion against exact integers, where its sums are longest
and its terms largest: digits and residues next to their moduli, moduli from a few units to 2^31."""
import random

import pytest

from grns_amd import largest_primes_below, product
from tests.helpers import to_res

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _primes_from(lo, n):
    from grns_amd.moduli import is_prime
    out, v = [], lo
    while len(out) < n:
        if is_prime(v):
            out.append(v)
        v += 1
    return out


def _sets(n):
    half = n // 2
    return {
        "near 2^31": largest_primes_below(n),
        "small": _primes_from(2, n),
        "near 2^16": _primes_from(1 << 16, n),
        "mixed": _primes_from(3, half) + largest_primes_below(n - half),
    }


@pytest.mark.parametrize("kind", ["near 2^31", "small", "near 2^16", "mixed"])
@pytest.mark.parametrize("n", [4, 8, 16, 32, 64])
def test_digit_edges(n, kind):
    import grns_amd as G
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mod = _sets(n)[kind]
    M = product(mod)
    rnd = random.Random(n)
    bases = [product(mod[:k]) for k in range(n)]
    vals = [0, 1, M - 1, M - 2, M // 2]
    vals += [b - 1 for b in bases[1:]] + bases + [M - b for b in bases]
    # every digit its modulus minus one, zero, or at random
    for _ in range(100):
        vals.append(sum(b * rnd.choice([0, m - 1, rnd.randrange(m)]) for b, m in zip(bases, mod)))
    vals += [rnd.randrange(M) for _ in range(200)]
    ctx = G.Context(mod, 0)
    got = ctx.mrc(torch.from_numpy(to_res(vals, mod)).cuda()).cpu().numpy()
    for j, v in enumerate(vals):
        want = []
        for m in mod:
            want.append(v % m)
            v //= m
        assert got[:, j].tolist() == want, (kind, j)
    # the digit arg-max on the same numbers
    res, idx = ctx.max(torch.from_numpy(to_res(vals, mod)).cuda(), mrc=True)
    assert int(idx.item()) == vals.index(max(vals))
    ctx.close()
