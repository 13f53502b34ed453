"""Division with a lane per pair (long arrays) against the wave-group form (the same pairs in short
calls) and exact integers: divisors of every length, quotients next to the digits' edges, remainders
next to 0 and to the divisor, partial waves, both layouts, operands written over, pairs left to the
reference loop, moduli counts between the padded sizes."""
import random

import numpy as np
import pytest

from grns_amd import largest_primes_below, product
from tests.helpers import to_res

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SHORT = 8000   # pairs per call of the wave-group form
LONG = 32768   # pairs of the lane form


def _set(name):
    n = int(name.split()[0])
    if "small" in name:
        return [v for v in range(2, 1000) if all(v % p for p in range(2, int(v ** 0.5) + 1))][:n]
    return largest_primes_below(n)


def _pairs(M, count, rnd):
    """(x, d): quotients and divisors around powers of 2^28, exact multiples and their neighbours."""
    L = M.bit_length()
    out = [(0, 1), (M - 1, 1), (M - 1, M - 1), (M - 2, M - 1), (M // 2, 2), (M - 1, 2), (1, M - 1)]
    while len(out) < count:
        d = max(1, min(M - 1, rnd.choice([
            rnd.getrandbits(rnd.randrange(1, L)), (1 << rnd.randrange(0, L - 1)) + rnd.randrange(-1, 2),
            (1 << 28 * rnd.randrange(0, (L - 1) // 28 + 1)) + rnd.randrange(-2, 3),
            ((1 << rnd.randrange(1, L)) - 1) << rnd.randrange(0, 28)])))
        top = (M - 1) // d
        q = min(top, rnd.choice([rnd.randrange(top + 1), rnd.getrandbits(rnd.randrange(1, L)),
                                 (1 << rnd.randrange(0, L)) + rnd.randrange(-1, 2),
                                 (rnd.getrandbits(20) << 28) | (1 << 27) + rnd.randrange(-2, 3)]))
        x = max(0, q) * d + rnd.choice([0, 1, d - 1, d // 2, rnd.randrange(d)])
        if 0 <= x < M:
            out.append((x, d))
    return out


def _short(ctx, x, d, fast):
    parts = [ctx.div(x[:, k:k + SHORT].contiguous(), d[:, k:k + SHORT].contiguous(), fast=fast)
             for k in range(0, x.shape[1], SHORT)]
    return torch.cat([q for q, _ in parts], 1), torch.cat([r for _, r in parts], 1)


@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("name", ["3", "8", "12 small", "16", "20", "32", "50", "64", "64 small"])
def test_div_lanes(name, fast):
    import grns_amd as G
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mod = _set(name)
    M, n = product(mod), len(mod)
    rnd = random.Random(n + fast)
    ctx = G.Context(mod, 0)
    base = _pairs(M, 2500, rnd)
    bx = torch.from_numpy(to_res([x for x, _ in base], mod)).cuda()
    bd = torch.from_numpy(to_res([d for _, d in base], mod)).cuda()
    keeps = np.array([[np.float64(m) * (1.0 / np.float64(m)) < 1.0] for m in mod])
    want_q = to_res([x // d for x, d in base], mod)
    want_q = np.where((want_q == 0) & keeps & np.array([[x >= d for x, d in base]]), np.array(mod)[:, None], want_q)
    want_r = to_res([x % d for x, d in base], mod)
    for extra in (0, 1, 63, 65):
        pick = torch.tensor([k % len(base) for k in range(LONG + extra)], device="cuda")
        x, d = bx[:, pick].contiguous(), bd[:, pick].contiguous()
        q, r = ctx.div(x, d, fast=fast)
        assert (q[:, :len(base)].cpu().numpy() == want_q).all()
        assert (r[:, :len(base)].cpu().numpy() == want_r).all()
        assert torch.equal(q, torch.from_numpy(want_q).cuda()[:, pick].to(torch.int32))
        assert torch.equal(r, torch.from_numpy(want_r).cuda()[:, pick].to(torch.int32))
    xn, dn = x.t().contiguous().t(), d.t().contiguous().t()
    qn, rn = ctx.div(xn, dn, fast=fast, q=torch.empty_like(xn), r=torch.empty_like(xn))
    assert qn.stride() == xn.stride() and torch.equal(qn, q) and torch.equal(rn, r)
    # results over the operands
    x2, d2 = x.clone(), d.clone()
    ctx.div(x2, d2, fast=fast, q=x2, r=d2)
    assert torch.equal(x2, q) and torch.equal(d2, r)
    # uniform dividends, and pairs for the reference loop: residues at or above m, zero divisors
    from grns_amd.workload import Synth
    syn = Synth(mod)
    x = syn.uniform(LONG + 77, 5, 1)
    x[:, :len(base)] = bx
    at = torch.arange(0, LONG, 97, device="cuda")
    if max(mod) < 1 << 30:
        x[n // 2, at] += mod[n // 2]
    dz = d[:, :1].expand(n, LONG + 77).clone()
    dz[:, :d.shape[1]] = d
    dz[:, 5::211] = 0
    q, r = ctx.div(x, dz, fast=fast)
    qs, rs = _short(ctx, x, dz, fast)
    ctx.status()
    assert torch.equal(q, qs) and torch.equal(r, rs)
    ctx.close()
