"""Scaling steps whose residues, or whose products with the rank weights, lie next to a multiple of
a modulus (where a step leaves its exact-division form), every partial exponent and small moduli,
against the CPU path; per call and in a batch plan."""
import random

import numpy as np
import pytest

from grns_amd import largest_primes_below, product
from tests.helpers import to_res

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _sets():
    primes = largest_primes_below(64)
    small = [v for v in range(3, 400) if all(v % p for p in range(2, int(v ** 0.5) + 1))]
    return {
        "8": largest_primes_below(8),
        "20": largest_primes_below(20),
        "64": primes,
        "small 32": small[:32],
        "mixed 12": small[20:26] + largest_primes_below(6),
    }


def _numbers(mod, count, seed):
    """x whose value after s steps of 2^30 has one residue (or rank product) within a few thousand of
    a multiple of its modulus, and an exponent that runs past that step."""
    rnd = random.Random(seed)
    M = product(mod)
    L = M.bit_length()
    xs, Ds = [], []
    while len(xs) < count:
        i = rnd.randrange(len(mod))
        m = mod[i]
        e = rnd.choice([-1, 1]) * rnd.choice([0, 1, 2, 1000, 2047, 2048, 2049, 4095, 4100, 6000, rnd.randrange(9000)])
        if rnd.random() < 0.5:
            e = e * (M // m)  # then (X w) mod m is the small value
        s = rnd.randrange(0, L // 30 + 1)
        top = M >> (30 * s)
        X = rnd.randrange(top + 1)
        X += (e - X) % m
        x = (X << (30 * s)) + rnd.randrange(1 << (30 * s))
        if x >= M:
            continue
        xs.append(x)
        Ds.append(30 * s + rnd.choice([0, 30, 60]) + rnd.randrange(0, 31))
    return xs, Ds


@pytest.mark.parametrize("name", list(_sets()))
def test_scale_step_edges(name):
    import grns_amd as G
    from oracle.oracle import Oracle
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mod = _sets()[name]
    ctx, orc = G.Context(mod, 0), Oracle(mod)
    xs, Ds = _numbers(mod, 1500, len(mod))
    x, D = to_res(xs, mod), np.array(Ds, np.uint32)
    want = orc.scale2pow_array(x, D)
    xd, Dd = torch.from_numpy(x).cuda(), torch.from_numpy(D.view(np.int32)).cuda()
    got = ctx.scale2pow(xd, Dd).cpu().numpy()
    assert (got == want).all()
    nm = ctx.scale2pow(xd.t().contiguous().t(), Dd).cpu().numpy()
    assert (nm == want).all()
    out = torch.zeros_like(xd)
    plan = G.Batch(ctx, [G.make_task("scale2pow", 700, a=xd[:, :700], out0=out[:, :700], D=Dd[:700]),
                         G.make_task("scale2pow", 800, a=xd[:, 700:], out0=out[:, 700:], D=Dd[700:])])
    plan.launch()
    assert (out.cpu().numpy() == want).all()
    plan.close()
    orc.close()
    ctx.close()
